"""Softmax over the last axis: the lanes of a row hold consecutive spans of it and its ordered sum
goes from lane to lane; few rows take a workgroup each, many a wave for 2 to 64 of them."""
import numpy as np
import pytest

import oracle
from tests import gpuops
from tests.helpers import assert_bit_exact, normal

pytestmark = pytest.mark.gpu


# lengths either side of where the rows of a wave halve and of whole fours; odd and even ones
@pytest.mark.parametrize("dim", [17, 18, 21, 31, 32, 33, 63, 64, 91, 127, 128, 129, 255, 256, 511, 512, 1022, 1023])
@pytest.mark.parametrize("rows", [1024, 1031, 4100])
def test_many_rows(gpu, rows, dim):
    x = normal(dim, rows * dim, 5.0)
    want = oracle.softmax(x, rows, dim, 1)
    assert_bit_exact(gpuops.softmax(x, rows, dim, 1, offset=rows % 4), want, "softmax")
    assert_bit_exact(gpuops.softmax(x, rows, dim, 1, inplace=True), want, "softmax in place")


# counts either side of 8192 waves of 64 and of 32 rows, and of 1024 waves of 32, 16, 8 and 4
@pytest.mark.parametrize("rows,dim", [(524287, 17), (524289, 20), (262143, 33), (262145, 40), (32767, 21), (32769, 21),
                                      (16383, 50), (16385, 96), (8191, 130), (8193, 140), (4095, 300), (4097, 300)])
def test_rows_of_a_wave(gpu, rows, dim):
    x = normal(rows % 97, rows * dim, 3.0)
    assert_bit_exact(gpuops.softmax(x, rows, dim, 1), oracle.softmax(x, rows, dim, 1), "softmax")


# a chunk of the workgroup form is 1024 elements, a lane's span 16
@pytest.mark.parametrize("dim", [1, 2, 3, 15, 16, 17, 64, 255, 1000, 1023, 1024, 1025, 1041, 2047, 2050, 15001])
@pytest.mark.parametrize("rows", [1, 3, 64, 1023])
def test_few_rows(gpu, rows, dim):
    x = normal(dim + rows, rows * dim, 5.0)
    assert_bit_exact(gpuops.softmax(x, rows, dim, 1, offset=dim % 4), oracle.softmax(x, rows, dim, 1), "softmax")


@pytest.mark.parametrize("rows,dim", [(1100, 21), (1100, 64), (1030, 700), (40, 21), (12, 1500)])
def test_rows_of_special_values(gpu, rows, dim):
    x = normal(9, rows * dim, 4.0).reshape(rows, dim).copy()
    x[1] = -np.inf
    x[2, dim - 1] = np.inf
    x[3, 0] = np.nan
    x[4, dim // 2] = np.nan
    x[5] = 3.0e38
    x[6] = -3.4028235e38
    x[7, ::2] -= 104.0  # underflow to zero and to subnormals, and subnormal quotients
    x[8, 1:] -= 88.0
    x[9, 1:] -= 100.0
    x[10] = 0.0
    with np.errstate(all="ignore"):
        want = oracle.softmax(x, rows, dim, 1)
        assert_bit_exact(gpuops.softmax(x, rows, dim, 1), want, "softmax")


# one to nine fours a lane, the last lane of a row with one element, a few and as many as the others; odd and even rows
@pytest.mark.parametrize("dim", [17, 20, 24, 25, 28, 33, 36, 37, 53, 56, 66, 79, 99, 131, 160, 201, 259, 272, 400, 515, 777, 992, 993, 1023])
@pytest.mark.parametrize("rows", [1025, 33003])
def test_last_lanes_of_rows(gpu, rows, dim):
    rows = min(rows, 4000000 // dim)
    x = normal(dim, rows * dim, 4.0)
    x[:dim] = -np.inf
    x[dim - 1] = 1.0
    x[3 * dim] = np.nan
    with np.errstate(all="ignore"):
        assert_bit_exact(gpuops.softmax(x, rows, dim, 1, offset=dim % 4), oracle.softmax(x, rows, dim, 1), "softmax")


# Rows longer than a chunk of 1024 of the ordered sum: a NaN in the first chunk and none behind it, sums that stay at a power of
# two, ties in every addition, and exponentials of all sizes; a workgroup a row in registers, and the longest beyond.
@pytest.mark.parametrize("dim", [1025, 2048, 3001, 4096, 8192, 9001])
def test_long_rows_of_special_sums(gpu, dim):
    rng = np.random.default_rng(dim)
    ln2 = np.log(2.0)
    kinds = [np.where(np.arange(dim) == 7, np.nan, rng.standard_normal(dim)),
             np.where(np.arange(dim) < dim // 2, 0.0, -25 * ln2),
             np.full(dim, -3.0),
             -ln2 * rng.integers(0, 27, dim),
             rng.uniform(-100.0, 0.0, dim),
             np.where(np.arange(dim) < 1024, 0.0, -24 * ln2),
             np.where(np.arange(dim) % 64 == 0, 0.0, -14 * ln2),
             np.where(np.arange(dim) == dim - 1, 80.0, rng.uniform(-20.0, 0.0, dim))]
    x = np.concatenate(kinds).astype(np.float32)
    with np.errstate(all="ignore"):
        want = oracle.softmax(x, len(kinds), dim, 1)
        assert_bit_exact(gpuops.softmax(x, len(kinds), dim, 1, offset=dim % 4), want, "softmax")


# a workgroup a row, in registers: one to eight vectors a lane, the last vector whole and cut, and the longest beyond
@pytest.mark.parametrize("dim", [5, 1022, 1028, 2045, 2048, 2049, 4093, 4096, 4097, 8189, 8190, 8192, 8193, 12000])
@pytest.mark.parametrize("rows", [1, 37])
def test_long_rows_of_a_workgroup(gpu, rows, dim):
    x = normal(dim, rows * dim, 4.0)
    if rows > 1:
        x[:dim] = -np.inf
        x[dim:2 * dim] = 1.0
        x[3 * dim - 1] = np.nan
        x[3 * dim:4 * dim] = -100.0
        x[4 * dim - 1] = 100.0
    with np.errstate(all="ignore"):
        want = oracle.softmax(x, rows, dim, 1)
        assert_bit_exact(gpuops.softmax(x, rows, dim, 1, offset=dim % 4), want, "softmax")
        assert_bit_exact(gpuops.softmax(x, rows, dim, 1, inplace=True), want, "softmax in place")
