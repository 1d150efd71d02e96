"""LRN with windows of one to seven channels: one, two or four waves of a workgroup share the channels of
64 positions, eight each, and hand the running sum on."""
import numpy as np
import pytest

import oracle
from tests import gpuops
from tests.helpers import assert_bit_exact, normal

pytestmark = pytest.mark.gpu


# channels either side of a round, of a span of four and of whole spans; positions either side of a wave
@pytest.mark.parametrize("channels", [3, 7, 8, 9, 10, 24, 31, 32, 33, 34, 63, 66, 97, 129])
@pytest.mark.parametrize("positions", [1, 63, 65, 130])
@pytest.mark.parametrize("size", [1, 3, 5, 7])
def test_lrn_spans(gpu, channels, positions, size):
    shape = (2, channels, 1, positions)
    x = normal(channels + size, 2 * channels * positions, 4.0)
    want = oracle.lrn(x, shape, size, 1e-2, 0.75, 1.0)[0]
    assert_bit_exact(gpuops.lrn(x, shape, size, 1e-2, 0.75, 1.0), want, "lrn")
    assert_bit_exact(gpuops.lrn(x, shape, size, 1e-2, 0.75, 1.0, inplace=True), want, "lrn in place")


@pytest.mark.parametrize("channels", [9, 35, 70])
def test_lrn_spans_of_special_values(gpu, channels):
    shape = (1, channels, 5, 30)
    x = normal(channels, channels * 150, 1.0).reshape(channels, 150).copy()
    x[channels // 2, :40] = np.inf
    x[0, 30:60] = np.nan
    x[channels - 1, 50:90] = 1e30
    x[:, 100:] = 0.0
    with np.errstate(all="ignore"):
        for k in (1.0, 0.0, -0.5):
            want = oracle.lrn(x, shape, 5, 1e-1, 0.75, k)[0]
            assert_bit_exact(gpuops.lrn(x, shape, 5, 1e-1, 0.75, k), want, "k = %g" % k)


# one, two and four waves for 64 positions: either side of 1280, 2560 and 3584 runs of 64, of 8, 16, 64 and 128 channels
@pytest.mark.parametrize("channels,positions", [(8, 3 * 27400), (17, 3 * 27305), (17, 3 * 27312), (33, 3 * 54612), (65, 3 * 54617), (9, 3 * 54700),
                                                (20, 3 * 76458), (20, 3 * 76461), (40, 3 * 76470), (137, 3 * 27400), (137, 3 * 54617)])
@pytest.mark.parametrize("size", [1, 5, 7])
def test_lrn_spans_of_many_positions(gpu, channels, positions, size):
    shape = (1, channels, 3, positions // 3)
    x = normal(channels + size, channels * positions, 4.0)
    want = oracle.lrn(x, shape, size, 1e-2, 0.75, 1.0)[0]
    assert_bit_exact(gpuops.lrn(x, shape, size, 1e-2, 0.75, 1.0), want, "lrn")
    assert_bit_exact(gpuops.lrn(x, shape, size, 1e-2, 0.75, 1.0, inplace=True), want, "lrn in place")


# two waves for 64 positions, 769 to 897 workgroups of 128: the ones beyond 768 cut in two where they are up to 128; several
# images, and a last run of one position
@pytest.mark.parametrize("images,positions", [(1, 98305), (3, 32789), (1, 114688), (1, 114689), (7, 14337)])
@pytest.mark.parametrize("channels,size", [(33, 5), (40, 3)])
def test_lrn_spans_cut_in_two(gpu, images, positions, channels, size):
    shape = (images, channels, 1, positions)
    x = normal(channels + size, images * channels * positions, 4.0)
    want = oracle.lrn(x, shape, size, 1e-2, 0.75, 1.0)[0]
    assert_bit_exact(gpuops.lrn(x, shape, size, 1e-2, 0.75, 1.0), want, "lrn")
    assert_bit_exact(gpuops.lrn(x, shape, size, 1e-2, 0.75, 1.0, inplace=True), want, "lrn in place")
