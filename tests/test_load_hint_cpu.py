"""Which accesses of device_common.h carry the non-temporal hint, read off the
gfx950 assembly of one kernel per helper, compiled with the library's flags."""
import re
import subprocess

import pytest

from shadow_amd import build

HELPERS = {  # helper -> (body, hint on the load, hint on the store)
    "load4_stream": ("q(y, load4_stream(x))", True, False),
    "load4_stream_any": ("q(y, load4_stream_any(x))", True, False),
    "load_stream": ("y[0] = load_stream(x)", True, False),
    "load4": ("q(y, load4(x))", False, False),
    "load4_any": ("q(y, load4_any(x))", False, False),
    "store4_stream": ("store4_stream(y, load4(x))", False, True),
    "store4_stream_any": ("store4_stream_any(y, load4(x))", False, True),
}


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    src = tmp_path_factory.mktemp("hint") / "hint.hip"
    text = ['#include "%s/device_common.h"' % build.CSRC, "using namespace shdw;",
            "SHDW_DEVICE void q(float* y, v4f v) { *reinterpret_cast<v4f*>(y) = v; }"]
    text += ['extern "C" __global__ void k_%s(const float* x, float* y) { x += 4 * threadIdx.x; y += 4 * threadIdx.x; %s; }'
             % (name, body) for name, (body, _, _) in HELPERS.items()]
    src.write_text("\n".join(text) + "\n")
    proc = subprocess.run([build.HIPCC] + build.HIP_FLAGS + ["--offload-device-only", "-S", str(src), "-o", "-"],
                          stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert proc.returncode == 0, proc.stderr
    return proc.stdout


@pytest.mark.parametrize("name", sorted(HELPERS))
def test_hints_of_the_access_helpers(assembly, name):
    """Streamed operands go past the caches in both directions, shared ones do not."""
    body = assembly.split("\nk_%s:" % name)[1].split("s_endpgm")[0]
    for what, hinted in (("load", HELPERS[name][1]), ("store", HELPERS[name][2])):
        lines = re.findall(r"global_%s_dword\S* [^\n]*" % what, body)
        assert len(lines) == 1, body
        assert bool(re.search(r"\bnt\b", lines[0])) is hinted, lines[0]
