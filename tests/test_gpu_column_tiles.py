"""Normalize and SSDNormalize on tiles of 64, 32 and 16 positions, whose column sums are taken in
any order where that cannot show: columns whose fp64 sum lies at the middle between two floats and
depends on the order, so that they have to be added front to back, next to columns that do not."""
import numpy as np
import pytest

import oracle
from tests import gpuops
from tests.helpers import assert_bit_exact, normal, uniform

F = np.float32
# (outer, dim, inner): one row more than the steps of the lanes, a last step with rows missing, whole
# tiles; positions that end one, two and three into a lane's four, on multiples of 4 and of 16
SHAPES = [(2, 65, 16), (1, 65, 4097), (3, 129, 37), (2, 255, 64), (2, 512, 100), (1, 511, 1444), (2, 513, 65), (1, 1024, 80),
          (2, 100, 67), (2, 128, 130), (3, 300, 46), (2, 600, 83), (1, 1000, 78)]


def tied_column(dim, squares):
    """Terms that add up front to back to exactly the middle between 1 and the next float (for the
    root of the sum with `squares`) and small ones that each are lost there, but not together."""
    c = np.zeros(dim, F)
    head = [F(1), F(2.0 ** -12), F(2.0 ** -12), F(2.0 ** -24)] if squares else [F(1), F(2.0 ** -24)]
    c[:len(head)] = head
    c[len(head):] = F(2.0 ** -27) if squares else F(2.0 ** -54)
    return c


def columns(outer, dim, inner, squares):
    x = normal(5, outer * dim * inner, 2.0).reshape(outer, dim, inner).copy()
    for s in {0, inner // 2, inner - 1}:
        x[:, :, s] = tied_column(dim, squares)
    return x


@pytest.mark.parametrize("squares", [False, True])
def test_the_sums_of_tied_columns_depend_on_the_order(squares):
    """The oracle's side: front to back gives 1 exactly, pairwise gives the next float."""
    c = tied_column(512, squares).astype(np.float64)
    t = c * c if squares else c
    front = np.float64(0)
    for v in t:
        front += v
    root = np.sqrt if squares else (lambda v: v)
    assert F(root(front)) == F(1)
    assert F(root(t[::-1].cumsum()[-1])) == np.nextafter(F(1), F(2))


@pytest.mark.gpu
@pytest.mark.parametrize("outer,dim,inner", SHAPES)
def test_sums_that_depend_on_the_order(gpu, outer, dim, inner):
    x = columns(outer, dim, inner, False)
    assert_bit_exact(gpuops.normalize(x, outer, dim, inner, 1.0, 1e-12), oracle.normalize(x, outer, dim, inner, 1.0, 1e-12), "p = 1")
    x = columns(outer, dim, inner, True)
    assert_bit_exact(gpuops.normalize(x, outer, dim, inner, 2.0, 1e-12), oracle.normalize(x, outer, dim, inner, 2.0, 1e-12), "p = 2")
    scale = uniform(6, dim, 0.5, 2.0)
    for eps in (0.0, 1e-10, -0.25):
        for sc, shared in ((scale, False), (scale[:1], True), (None, True)):
            want = oracle.ssd_normalize(x, outer, dim, inner, False, shared, eps, sc)
            assert_bit_exact(gpuops.ssd_normalize(x, outer, dim, inner, False, shared, eps, sc, offset=1), want, "eps %g" % eps)


@pytest.mark.gpu
@pytest.mark.parametrize("outer,dim,inner", SHAPES)
def test_zeros_infinities_and_nans_in_columns(gpu, outer, dim, inner):
    x = normal(7, outer * dim * inner, 2.0).reshape(outer, dim, inner).copy()
    x[:, :, 1] = 0.0
    x[:, dim - 1, 2] = np.inf
    x[:, 0, 3] = np.nan
    x[:, :, 4] *= F(1e-30)
    x[:, :, 5] *= F(1e25)
    x[:, :, 6] = -np.inf
    with np.errstate(all="ignore"):
        for p in (1.0, 2.0):
            for eps in (1e-12, 0.0):
                want = oracle.normalize(x, outer, dim, inner, p, eps)
                assert_bit_exact(gpuops.normalize(x, outer, dim, inner, p, eps), want, "p = %g, eps %g" % (p, eps))
        want = oracle.ssd_normalize(x, outer, dim, inner, False, True, 1e-10, None)
        assert_bit_exact(gpuops.ssd_normalize(x, outer, dim, inner, False, True, 1e-10, None), want, "ssd")
        assert_bit_exact(gpuops.softmax(x, outer, dim, inner), oracle.softmax(x, outer, dim, inner), "softmax")


def whole_columns(outer, dim, inner, largest):
    """Whole numbers, every third column's sum made odd and past 2^24: exactly between two floats or next to it."""
    x = np.random.default_rng(11).integers(0, largest, (outer, dim, inner)).astype(F)
    over = np.sum(x, axis=1, dtype=np.float64)
    x[:, 7, ::3] += ((1 + np.float64(1 << 24) - over[:, ::3]).clip(0) // 2 * 2 + (over[:, ::3] + 1) % 2).astype(F)
    x[:, dim - 1, ::5] = 0
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("outer,dim,inner", SHAPES)
def test_sums_that_are_exact_in_any_order(gpu, outer, dim, inner):
    """Alone and beside columns that have to be added in order."""
    for largest in (2, 256, 1 << 18):
        x = whole_columns(outer, dim, inner, largest)
        for y in (x, np.where(np.arange(inner) % 16 == 3, tied_column(dim, False)[:, None], x).astype(F)):
            want = oracle.normalize(y, outer, dim, inner, 1.0, 1e-12)
            assert_bit_exact(gpuops.normalize(y, outer, dim, inner, 1.0, 1e-12), want, "p = 1, below %d" % largest)
        y = np.sqrt(x).astype(F) if largest == 2 else x
        want = oracle.normalize(y, outer, dim, inner, 2.0, 1e-12)
        assert_bit_exact(gpuops.normalize(y, outer, dim, inner, 2.0, 1e-12), want, "p = 2, below %d" % largest)


@pytest.mark.gpu
@pytest.mark.parametrize("outer,dim,inner", SHAPES)
def test_negative_eps_next_to_the_sum(gpu, outer, dim, inner):
    """sum + eps is 0, negative or a few last places of the sum."""
    x = columns(outer, dim, inner, True)
    x[:, :, 1::2] = F(2.0 ** -5)
    eps = dim * 2.0 ** -10
    with np.errstate(all="ignore"):
        for e in (-1.0, -eps, -eps * (1 + 2.0 ** -20), -eps * (1 - 2.0 ** -20), -1e9):
            want = oracle.ssd_normalize(x, outer, dim, inner, False, True, e, None)
            assert_bit_exact(gpuops.ssd_normalize(x, outer, dim, inner, False, True, e, None), want, "eps %g" % e)


# a factor a row on tall tiles: up to 512 of them take the factors through LDS
@pytest.mark.gpu
@pytest.mark.parametrize("outer,dim,inner", [(1, 513, 8192), (1, 513, 8193), (2, 700, 4094), (3, 1024, 77), (1, 951, 1681), (2, 1023, 64), (2, 601, 4112)])
def test_factors_of_tall_tiles(gpu, outer, dim, inner):
    x = normal(8, outer * dim * inner, 2.0)
    scale = uniform(9, dim, 0.5, 2.0)
    want = oracle.ssd_normalize(x, outer, dim, inner, False, False, 1e-10, scale)
    assert_bit_exact(gpuops.ssd_normalize(x, outer, dim, inner, False, False, 1e-10, scale), want, "ssd")
    assert_bit_exact(gpuops.ssd_normalize(x, outer, dim, inner, False, False, 1e-10, scale, inplace=True, offset=1), want, "ssd in place")
