"""How Softmax's tile kernel cuts a shape (shadow_amd/csrc/softmax_shape.h): what every cut has to keep to,
and which form the shapes of the GPU tests and of its rules get."""
import ctypes
import os

import pytest

from tests.native import build

HERE = os.path.dirname(os.path.abspath(__file__))
POSITIONS, SLOTS, PASSES = {6, 5, 4}, {8, 10, 16}, {1, 2}


@pytest.fixture(scope="module")
def native():
    path = os.path.join(HERE, "native", "softmax_shape.so")
    if not os.path.exists(path):
        build.build()
    return ctypes.CDLL(path)


def cut(native, outer, dim, inner, sectors):
    out = (ctypes.c_uint * 5)()
    native.softmax_tiles(outer, dim, inner, int(sectors), out)
    shift, slots, grid, passes, lds = out
    return {"form": (shift, slots, passes), "grid": grid, "lds": lds}


@pytest.mark.parametrize("sectors", [0, 1])
@pytest.mark.parametrize("inner", [16, 17, 64, 65, 361, 1444, 3136, 5184, 16384, 65536])
def test_every_cut_fits_the_kernel(native, inner, sectors):
    for outer in (1, 2, 5, 16, 33, 64, 100, 257, 769, 1025, 1793):
        if outer * inner * 1024 < 2 ** 31:
            assert native.softmax_tiles_scan(outer, inner, sectors) == 0, outer


def test_forms_of_the_gpu_shapes(native):
    """The shapes of test_gpu_softmax_tiles.py get the forms they are there for, each with all three kinds of rows."""
    from tests.test_gpu_softmax_tiles import CUTS, offset
    reached = set()
    for (outer, dim, inner), form in CUTS.items():
        sectors = inner % 16 == 0 and offset(dim) == 0
        assert cut(native, outer, dim, inner, sectors)["form"] == form, (outer, dim, inner)
        reached.add((form, "sectors" if sectors else "quads" if inner % 4 == 0 else "any"))
    forms = {(s, n, p) for s in POSITIONS for n in SLOTS for p in PASSES} - {(4, 8, 2)}
    assert reached == {(f, rows) for f in forms for rows in ("sectors", "quads", "any")}


# Two passes where LDS holds the tiles a CU down, and all tiles are on the chip at once with them; not where registers do
# (columns of 65 to 86 of eight vectors), nor where there are more rounds of tiles than one.
@pytest.mark.parametrize("shape,sectors,form", [
    ((64, 70, 12544), True, (6, 8, 1)), ((64, 86, 12544), True, (6, 8, 1)), ((32, 91, 5184), True, (6, 8, 1)), ((64, 100, 3136), True, (6, 8, 1)),
    ((1700, 86, 64), True, (6, 8, 1)), ((1700, 87, 64), True, (6, 8, 2)), ((16, 91, 6400), True, (6, 8, 2)), ((64, 128, 5000), False, (6, 8, 1)),
    ((16, 150, 5184), True, (6, 10, 2)), ((64, 150, 5184), True, (6, 10, 1)), ((158, 150, 1605), False, (6, 10, 1)), ((62, 150, 1605), False, (6, 10, 2)),
    ((123, 640, 405), False, (4, 10, 1)), ((68, 320, 805), False, (5, 10, 1)), ((68, 320, 800), True, (5, 10, 2)), ((62, 640, 405), False, (4, 10, 1)),
    ((62, 1000, 405), False, (4, 16, 2)), ((16, 500, 1600), True, (5, 16, 2)), ((1, 150, 5184), True, (5, 8, 1))])
def test_passes(native, shape, sectors, form):
    assert cut(native, *shape, sectors)["form"] == form


# 64, 32 and 16 positions: few tiles are halved, and once more where the last of 32 would have one to four
@pytest.mark.parametrize("shape,shift", [
    ((43, 71, 96), 5), ((43, 71, 97), 4), ((43, 71, 100), 4), ((43, 71, 101), 5), ((43, 71, 128), 5), ((109, 71, 100), 4), ((110, 71, 100), 5), ((111, 71, 96), 5),
    ((200, 71, 100), 6), ((43, 200, 100), 4), ((200, 200, 100), 4), ((300, 200, 100), 5), ((500, 200, 100), 6), ((43, 200, 104), 5), ((4, 300, 100), 4)])
def test_positions(native, shape, shift):
    assert cut(native, *shape, False)["form"][0] == shift


def test_lds_of_the_gpu_shapes(native):
    """The rows of a pass, the exponentials' table and a tile row for each of four waves."""
    for (outer, dim, inner), lds in {(400, 100, 65): 100 * 256 + 256 + 1024, (520, 127, 65): 64 * 256 + 256 + 1024,
                                     (400, 160, 80): 96 * 256 + 256 + 1024, (180, 512, 65): 256 * 128 + 256 + 512,
                                     (8, 512, 68): 512 * 64 + 256 + 256, (104, 1024, 65): 512 * 64 + 256 + 256}.items():
        assert cut(native, outer, dim, inner, False)["lds"] == lds, (outer, dim, inner)
