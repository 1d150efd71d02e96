"""The fp32 running sum by a whole wave (shadow_amd/csrc/ordered_sum.h), modelled lane by lane: the bits of the
additions in turn for every number of terms a lane that kernels take, any incoming sum, and terms whose sums pass
powers of two in every way; guesses of the power of two that were wrong are among them, and found out."""
import ctypes
import os

import pytest

from tests.native import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def native():
    path = os.path.join(HERE, "native", "ordered_sum.so")
    if not os.path.exists(path):
        build.build()
    lib = ctypes.CDLL(path)
    lib.ordered_sum_scan.restype = ctypes.c_long
    lib.ordered_sum_near.restype = ctypes.c_long
    for fn in (lib.ordered_sum_scan, lib.ordered_sum_near):
        fn.argtypes = [ctypes.c_int, ctypes.c_uint, ctypes.c_long, ctypes.POINTER(ctypes.c_long)]
    return lib


@pytest.mark.parametrize("seed", [1, 2, 3])
@pytest.mark.parametrize("terms", [16, 28, 32])  # Softmax's rows, the gated block's, whole-plane averages
def test_sums_of_a_wave_are_the_running_sums(native, terms, seed):
    counts = (ctypes.c_long * 3)()
    assert native.ordered_sum_scan(terms, seed, 20000, counts) == 0
    wrong, one_by_one, joined_anew = counts
    assert wrong > 1000 and one_by_one > 20000 and joined_anew > 1000


@pytest.mark.parametrize("terms", [16, 28, 32])
def test_a_wrong_guess_leaves_few_lanes_to_add_one_by_one(native, terms):
    """Sums that pass a power of two within rounding of a lane's end, any lane: what is left of the run is joined anew."""
    counts = (ctypes.c_long * 4)()
    assert native.ordered_sum_near(terms, 7, 4000, counts) == 0
    wrong, one_by_one, joined_anew, most = counts
    assert wrong > 400 and joined_anew > 400
    assert one_by_one < 9 * 4000  # the lanes that a sum passes powers of two in, about six
    assert most <= 10  # of any chunk: those, and two or three more for a wrong guess
