"""Softmax over columns of 65 to 1024 on tiles of 64, 32 and 16 positions: every size of a lane's share,
whole columns in LDS and two passes, positions in whole sectors, whole quads and neither."""
import ctypes

import numpy as np
import pytest

import oracle
import shadow_amd
from tests import gpuops
from tests.helpers import assert_bit_exact, normal, with_specials

pytestmark = pytest.mark.gpu

# (outer, dim, inner, log2 of the positions): in this order half the positions, eight vectors a lane, one pass
# and two; 64 positions, ten vectors, one pass and two, and sixteen; 32, ten, one pass and two, and sixteen
# likewise; 16 of eight; 16 of ten, one pass and two, and sixteen likewise
CUTS = [(1, 65, 64, 5), (2, 160, 100, 5), (8, 161, 130, 5), (8, 256, 80, 5), (350, 256, 65, 5),
        (400, 100, 65, 6), (400, 160, 65, 6), (400, 160, 80, 6), (400, 159, 68, 6), (600, 200, 65, 6),
        (160, 300, 65, 5), (260, 320, 65, 5), (160, 321, 65, 5), (180, 512, 65, 5),
        (2, 257, 66, 4), (8, 512, 68, 4),
        (5, 513, 65, 4), (155, 640, 65, 4), (3, 641, 65, 4), (2, 1024, 80, 4), (104, 1024, 65, 4)]


@pytest.mark.parametrize("outer,dim,inner,shift", CUTS)
def test_softmax_tiles(gpu, outer, dim, inner, shift):
    path, variant = ctypes.c_int(), ctypes.c_int()
    assert shadow_amd.hip().shdw_hip_softmax_plan(outer, dim, inner, ctypes.byref(path), ctypes.byref(variant), None) == 0
    assert variant.value == shift
    x = normal(dim, outer * dim * inner, 3.0)
    first = x[:dim * inner].reshape(dim, inner)
    first[:] = with_specials(first.ravel(), 3).reshape(dim, inner)
    first[:, inner // 2] = -np.inf
    first[0, inner // 2] = 5.0
    with np.errstate(all="ignore"):
        want = oracle.softmax(x, outer, dim, inner)
        assert_bit_exact(gpuops.softmax(x, outer, dim, inner, inplace=dim % 2 == 1, offset=dim % 3), want, "softmax")
