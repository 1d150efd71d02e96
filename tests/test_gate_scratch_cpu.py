"""The gated block's kernels hold their rows in registers: what the compiler says of each form's scratch memory."""
import os
import re
import subprocess

from shadow_amd import build


def test_no_form_of_the_gated_block_spills():
    cmd = [build.HIPCC] + build.HIP_FLAGS + ["-Rpass-analysis=kernel-resource-usage", "--offload-device-only", "-c",
                                             os.path.join(build.CSRC, "gate.hip"), "-o", os.devnull]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert proc.returncode == 0, proc.stdout
    names = re.findall(r"Function Name: (\S*squeeze_gate_kernel\S*)", proc.stdout)
    scratch = [int(v) for v in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", proc.stdout)]
    assert len(names) == len(scratch) >= 12
    assert not any(scratch), [(n, s) for n, s in zip(names, scratch) if s]
