"""The gated block's kernels and the row softmax hold their rows in registers: what the compiler says of each form's
scratch memory, and of the waves that a SIMD has room for."""
import functools
import os
import re
import subprocess

from shadow_amd import build


@functools.lru_cache(maxsize=None)
def remarks(source="gate.hip"):
    cmd = [build.HIPCC] + build.HIP_FLAGS + ["-Rpass-analysis=kernel-resource-usage", "--offload-device-only", "-c",
                                             os.path.join(build.CSRC, source), "-o", os.devnull]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert proc.returncode == 0, proc.stdout
    return proc.stdout


def test_no_form_of_the_gated_block_spills():
    names = re.findall(r"Function Name: (\S*squeeze_gate_kernel\S*)", remarks())
    scratch = [int(v) for v in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", remarks())]
    assert len(names) == len(scratch) >= 12
    assert not any(scratch), [(n, s) for n, s in zip(names, scratch) if s]


def test_waves_that_four_vectors_of_a_row_leave_room_for():
    """1675 workgroups of them fit 256 CUs at once as seven a CU; as six, a few are left for a second round."""
    names = re.findall(r"Function Name: (\S*squeeze_gate_kernel\S*)", remarks())
    waves = [int(v) for v in re.findall(r"Occupancy \[waves/SIMD\]: (\d+)", remarks())]
    assert len(names) == len(waves)
    # four vectors, whole vectors or not, whole in LDS, one row a lane; and whole rows of up to four vectors a lane, 14000 rows of
    # 448 with 32 lanes each 8.5 us, 12.5 as six
    forms = {n: w for n, w in zip(names, waves)
             if re.search(r"19squeeze_gate_kernelILi4ELb[01]ELb1ELb1E|whole_squeeze_gate_kernelILi[1-4]E", n)}
    assert len(forms) >= 12 + 8
    assert min(forms.values()) >= 7, forms


def test_waves_that_eight_vectors_of_a_softmax_row_leave_room_for():
    said = remarks("softmax.hip").split("Function Name: ")[1:]
    forms = [f for f in said if re.match(r"\S*softmax_row_kernelILi8E", f)]
    assert len(forms) == 1
    assert int(re.search(r"Occupancy \[waves/SIMD\]: (\d+)", forms[0]).group(1)) >= 7
    assert int(re.search(r"ScratchSize \[bytes/lane\]: (\d+)", forms[0]).group(1)) == 0
