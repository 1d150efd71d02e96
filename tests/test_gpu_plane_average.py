"""Whole-plane averages of 256 and more elements: the sum of a plane goes from lane to lane, 32
elements each, in chunks of 32 * 64 / G columns for G = 1, 2, 4 or 8 planes a wave."""
import numpy as np
import pytest

import oracle
from tests import gpuops
from tests.helpers import assert_bit_exact, normal, with_specials

pytestmark = pytest.mark.gpu

# planes either side of where G changes (1024, 2048, 4096) and of whole waves and workgroups;
# lengths either side of a lane's span, of a chunk and of whole vectors
PLANES = [1, 3, 1023, 1025, 2047, 2050, 4095, 4097, 4129]
LENGTHS = [256, 257, 287, 289, 511, 514, 1023, 1027, 2048, 2049, 4099]


@pytest.mark.parametrize("length", LENGTHS)
@pytest.mark.parametrize("planes", PLANES)
def test_whole_plane_average(gpu, planes, length):
    x = normal(planes + length, planes * length, 2.0)
    shape, out = (1, planes, 1, length), (1, planes, 1, 1)
    want = oracle.pooling(x, shape, 1, (1, length), (1, 1), (0, 0), out)
    assert_bit_exact(gpuops.pooling(x, shape, 1, (1, length), (1, 1), (0, 0), out, offset=planes % 4), want, "average")


@pytest.mark.parametrize("length", [256, 515, 2051])
def test_whole_plane_average_of_special_values(gpu, length):
    shape, out = (5, 7, length), (5, 7, 1)
    x = with_specials(normal(3, 35 * length, 2.0), 3).reshape(shape)
    x[1] = -0.0
    x[2] = np.float32(1e-42)
    x[3, :, -1] = np.inf
    args = ((5, 7, 1, length), 1, (1, length), (1, 1), (0, 0), (5, 7, 1, 1))
    with np.errstate(all="ignore"):
        assert_bit_exact(gpuops.pooling(x, *args), oracle.pooling(x, *args), "average")


def settles_near_one(rng, length):
    """Stays within rounding of a power of two for lanes on end: whether a sum has passed it depends on the order."""
    head = rng.random(int(rng.integers(33, 600)))
    x = np.zeros(length)
    x[:head.size] = head / head.sum()
    x[head.size:] = np.ldexp(rng.random(length - head.size), -30)
    return x


def reaches_a_power_at_a_lanes_end(rng, length):
    """The sum is a power of two, but for rounding, where a lane's 16, 28 or 32 terms end: guesses of it differ."""
    x = rng.random(length)
    end = int(rng.choice([16, 28, 32])) * int(rng.integers(3, 36))
    total = x[:end].sum()
    return x * (2.0 ** np.floor(np.log2(total)) / total)


def rows_without_signs(seed, planes, length):
    """Rows whose running sums pass powers of two in every way: sums that grow evenly, ties in
    every addition, terms of all sizes, subnormal sums, sums that overflow, and a sign somewhere."""
    rng = np.random.default_rng(seed)
    x = np.maximum(rng.standard_normal((planes, length)), 0).astype(np.float32)
    kinds = [lambda: np.full(length, 1.0),
             lambda: np.ldexp(1.0, rng.integers(-24, 1, length)),                  # ties
             lambda: np.ldexp(rng.random(length), rng.integers(-40, 41, length)),
             lambda: np.ldexp(rng.integers(0, 9, length).astype(float), -149),     # subnormal all the way
             lambda: rng.random(length) * 3e38,                                    # overflows
             lambda: np.where(np.arange(length) < length // 2, 0.0, rng.random(length)),
             lambda: np.where(np.arange(length) == 3 * length // 4, -50.0, rng.random(length)),
             lambda: np.where(np.arange(length) == length - 1, np.inf, 0.1),
             lambda: np.where(np.arange(length) == 40, -0.0, rng.random(length)),
             lambda: np.where(np.arange(length) == 1, np.nan, 1.0),
             lambda: np.where(np.arange(length) % 64 == 0, 2.0 ** 24, 1.0),
             lambda: np.where(np.arange(length) == 0, 2.0 ** 24 - 1, 0.5),
             lambda: settles_near_one(rng, length),
             lambda: reaches_a_power_at_a_lanes_end(rng, length),
             lambda: reaches_a_power_at_a_lanes_end(rng, length)]
    for r in range(min(planes, 30 * len(kinds))):
        x[r] = kinds[r % len(kinds)]()
    return x


# lengths either side of where the additions are taken side by side, of a chunk, of a lane's span
# and of whole vectors; planes either side of the most that a wave each is taken for
@pytest.mark.parametrize("length", [1151, 1152, 1155, 2016, 2047, 2048, 2049, 4098, 6211])
@pytest.mark.parametrize("planes", [60, 2048, 2049])
def test_whole_plane_average_without_signs(gpu, planes, length):
    x = rows_without_signs(planes + length, planes, length)
    args = ((1, planes, 1, length), 1, (1, length), (1, 1), (0, 0), (1, planes, 1, 1))
    with np.errstate(all="ignore"):
        want = oracle.pooling(x, *args)
        assert_bit_exact(gpuops.pooling(x, *args, offset=length % 4), want, "average")
