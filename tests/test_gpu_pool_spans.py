"""2-D pooling through LDS bands that are held as they lie in memory: rows of any width, or off the
vector boundary, with windows that need no cells beside the rows."""
import ctypes

import pytest

import oracle
import shadow_amd
from tests import gpuops
from tests.helpers import assert_bit_exact, normal

pytestmark = pytest.mark.gpu

BAND = 24


# width, kernel, stride, vertical padding: odd widths, multiples of four off the boundary, spans that are no
# whole vectors, last bands shorter than the others, windows that hang over the last row
@pytest.mark.parametrize("h,w,kernel,stride,pad_h,over", [
    (55, 55, (3, 3), (2, 2), 0, 0), (57, 61, (2, 2), (2, 2), 0, 0), (77, 99, (7, 7), (4, 4), 3, 0), (131, 67, (3, 5), (3, 2), 1, 0),
    (40, 257, (5, 5), (3, 3), 0, 0), (200, 64, (2, 2), (2, 2), 0, 0), (56, 64, (3, 3), (1, 3), 1, 0), (90, 91, (4, 3), (4, 4), 0, 1),
    (300, 15, (3, 3), (3, 3), 0, 0), (64, 1001, (2, 3), (2, 2), 0, 0)])
@pytest.mark.parametrize("pool_type", [0, 1])
@pytest.mark.parametrize("offset", [0, 1, 2])
def test_pooling_over_spans(gpu, h, w, kernel, stride, pad_h, over, pool_type, offset):
    n, c = 3, 5
    oh = (h + 2 * pad_h - kernel[0]) // stride[0] + 1 + over
    ow = (w - kernel[1]) // stride[1] + 1
    shape, out = [n, c, h, w], [n, c, oh, ow]
    x = normal(h + w, n * c * h * w, 2.0)
    want = oracle.pooling(x, shape, pool_type, kernel, stride, (pad_h, 0), out)
    assert_bit_exact(gpuops.pooling(x, shape, pool_type, kernel, stride, (pad_h, 0), out, offset=offset), want, "pooling")


def test_the_spans_are_bands(gpu):
    path = ctypes.c_int()
    for h, w in ((55, 55), (90, 91)):
        o = [(h - 3) // 2 + 1, (w - 3) // 2 + 1]
        shadow_amd.check(shadow_amd.hip().shdw_hip_pooling2d_plan(shadow_amd.ints([3, 5, h, w]), 0, 3, 3, 2, 2, 0, 0,
                                                                  shadow_amd.ints([3, 5] + o), ctypes.byref(path), None, None))
        assert path.value == BAND
