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
TILE = 9  # SHDW_PATH_TILE

# (outer, dim, inner): (log2 of a tile's positions, vectors a lane has room for, passes through LDS), as
# tests/test_softmax_shape_cpu.py has it: every form that is launched, its rows in whole sectors, whole quads and neither
CUTS = {
    (257, 65, 68): (6, 8, 1), (257, 66, 80): (6, 8, 1), (400, 100, 65): (6, 8, 1), (520, 126, 80): (6, 8, 2),
    (520, 127, 65): (6, 8, 2), (520, 127, 68): (6, 8, 2), (257, 129, 65): (6, 10, 1), (257, 129, 68): (6, 10, 1),
    (257, 129, 80): (6, 10, 1), (400, 159, 68): (6, 10, 2), (400, 159, 80): (6, 10, 2), (400, 160, 65): (6, 10, 2),
    (400, 160, 80): (6, 10, 2), (700, 161, 65): (6, 16, 1), (700, 161, 68): (6, 16, 1), (700, 162, 80): (6, 16, 1),
    (600, 161, 68): (6, 16, 2), (600, 162, 80): (6, 16, 2), (600, 200, 65): (6, 16, 2), (1, 65, 64): (5, 8, 1),
    (1, 66, 64): (5, 8, 1), (2, 160, 108): (5, 8, 1), (8, 161, 139): (5, 8, 1), (8, 256, 80): (5, 8, 1),
    (350, 255, 76): (5, 8, 2), (350, 255, 80): (5, 8, 2), (350, 256, 70): (5, 8, 2), (155, 257, 68): (5, 10, 1),
    (155, 258, 80): (5, 10, 1), (160, 300, 65): (5, 10, 1), (257, 318, 80): (5, 10, 2), (257, 319, 68): (5, 10, 2),
    (260, 320, 65): (5, 10, 2), (160, 321, 65): (5, 16, 1), (155, 321, 68): (5, 16, 1), (155, 321, 80): (5, 16, 1),
    (257, 321, 68): (5, 16, 2), (257, 321, 80): (5, 16, 2), (180, 512, 65): (5, 16, 2), (43, 71, 97): (4, 8, 1),
    (2, 160, 100): (4, 8, 1), (8, 161, 130): (4, 8, 1), (43, 200, 100): (4, 8, 1), (200, 250, 100): (4, 8, 1),
    (350, 255, 68): (4, 8, 1), (350, 256, 65): (4, 8, 1), (2, 257, 66): (4, 8, 1), (1, 258, 64): (4, 8, 1),
    (8, 512, 68): (4, 8, 1), (5, 513, 65): (4, 10, 1), (1, 513, 68): (4, 10, 1), (1, 513, 64): (4, 10, 1),
    (155, 639, 68): (4, 10, 2), (155, 639, 80): (4, 10, 2), (155, 640, 65): (4, 10, 2), (3, 641, 65): (4, 16, 1),
    (1, 641, 68): (4, 16, 1), (1, 642, 64): (4, 16, 1), (2, 1024, 80): (4, 16, 1), (155, 641, 68): (4, 16, 2),
    (155, 642, 80): (4, 16, 2), (104, 1024, 65): (4, 16, 2),
}


def offset(dim):
    """Floats that x and y are off the vector boundary."""
    return dim % 3


@pytest.mark.parametrize("outer,dim,inner", CUTS)
def test_softmax_tiles(gpu, outer, dim, inner):
    path, variant = ctypes.c_int(), ctypes.c_int()
    assert shadow_amd.hip().shdw_hip_softmax_plan(outer, dim, inner, ctypes.byref(path), ctypes.byref(variant), None) == 0
    assert (path.value, variant.value) == (TILE, CUTS[outer, dim, inner][0])
    x = normal(dim, outer * dim * inner, 3.0)
    first = x[:dim * inner].reshape(dim, inner)
    first[:] = with_specials(first.ravel(), 3).reshape(dim, inner)
    first[:, inner // 2] = -np.inf
    first[0, inner // 2] = 5.0
    with np.errstate(all="ignore"):
        want = oracle.softmax(x, outer, dim, inner)
        assert_bit_exact(gpuops.softmax(x, outer, dim, inner, inplace=dim % 2 == 1, offset=offset(dim)), want, "softmax")
