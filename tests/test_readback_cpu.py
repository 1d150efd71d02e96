"""Reading results back (shdw_hip_memcpy_d2h_staged, the allocator's read): which sources go by
the copy kernel and which by the runtime's copy, on a HIP runtime made for the test
(tests/native/readback.cpp)."""
import os
import subprocess

from tests.native import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_kernel_reads_only_what_it_can_reach():
    """Memory that no kernel of the device reaches, or a range past its allocation, goes to the runtime's copy, which
    checks; failing to get pinned memory leaves no error behind."""
    exe = os.path.join(HERE, "native", "readback")
    if not os.path.exists(exe):
        build.build()
    out = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.count("ok ") == 12, out.stdout
