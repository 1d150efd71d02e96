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


# the same on rows of a multiple of four columns off the boundary, walked four outputs at a time
@pytest.mark.parametrize("h,w,kernel", [(64, 64, (3, 3)), (40, 120, (5, 5)), (50, 32, (2, 4)), (90, 76, (3, 5))])
@pytest.mark.parametrize("pool_type", [0, 1])
def test_pooling_over_spans_at_stride_one(gpu, h, w, kernel, pool_type):
    n, c = 3, 5
    shape, out = [n, c, h, w], [n, c, h - kernel[0] + 1, w - kernel[1] + 1]
    x = normal(h + w, n * c * h * w, 2.0)
    want = oracle.pooling(x, shape, pool_type, kernel, (1, 1), (0, 0), out)
    for offset in (1, 3):
        assert_bit_exact(gpuops.pooling(x, shape, pool_type, kernel, (1, 1), (0, 0), out, offset=offset), want, "pooling")


def band_variant(shape, k, stride, pad, pool_type=0):
    """Of a band: 100 x vectors a lane for rows of vectors, 10 x for spans, 0 for single floats; and the output's shape."""
    out = shape[:2] + [(s + 2 * pad - k) // stride + 1 for s in shape[2:]]
    path, variant = ctypes.c_int(), ctypes.c_int()
    shadow_amd.check(shadow_amd.hip().shdw_hip_pooling2d_plan(shadow_amd.ints(shape), pool_type, k, k, stride, stride, pad, pad,
                                                              shadow_amd.ints(out), ctypes.byref(path), ctypes.byref(variant), None))
    assert path.value == BAND
    return variant.value, out


# vectors, spans and single floats, either side of 24 MB of input and with and without rows that bands share:
# every kind of loads and stores that a band has
@pytest.mark.parametrize("shape,k,stride,pad,least,most", [
    ([3, 5, 160, 160], 5, 3, 0, 100, 999), ([9, 56, 112, 112], 2, 1, 0, 100, 999), ([9, 56, 112, 112], 4, 4, 0, 100, 999),
    ([9, 56, 112, 112], 5, 2, 0, 100, 999), ([3, 5, 57, 61], 2, 2, 0, 20, 99), ([9, 56, 113, 113], 2, 2, 0, 20, 99),
    ([9, 56, 113, 113], 3, 2, 0, 20, 99), ([3, 5, 55, 55], 3, 2, 1, 0, 9), ([9, 56, 113, 113], 3, 2, 1, 0, 9), ([4, 8, 450, 451], 3, 2, 1, 0, 9)])
@pytest.mark.parametrize("pool_type", [0, 1])
def test_every_kind_of_band(gpu, shape, k, stride, pad, least, most, pool_type):
    variant, out = band_variant(shape, k, stride, pad, pool_type)
    assert least <= variant <= most
    n = shape[0] * shape[1] * shape[2] * shape[3]
    x = normal(k + stride, n, 2.0)
    want = oracle.pooling(x, shape, pool_type, (k, k), (stride, stride), (pad, pad), out)
    assert_bit_exact(gpuops.pooling(x, shape, pool_type, (k, k), (stride, stride), (pad, pad), out), want, "pooling")


def test_the_spans_are_bands(gpu):
    path = ctypes.c_int()
    for h, w in ((55, 55), (90, 91)):
        o = [(h - 3) // 2 + 1, (w - 3) // 2 + 1]
        shadow_amd.check(shadow_amd.hip().shdw_hip_pooling2d_plan(shadow_amd.ints([3, 5, h, w]), 0, 3, 3, 2, 2, 0, 0,
                                                                  shadow_amd.ints([3, 5] + o), ctypes.byref(path), None, None))
        assert path.value == BAND
