"""Transpositions with a thin side, whose tiles get shorter where there are few of them: long sides that end
inside a tile and inside a vector, in both directions."""
import numpy as np
import pytest

from shadow_amd import Buffer, check, hip, ints
from tests.helpers import normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("thin", [1, 2, 3, 8, 15, 16, 65, 72, 84, 126, 127])
@pytest.mark.parametrize("batch,big", [(1, 256), (1, 257), (3, 361), (16, 290), (20, 1444), (2, 5003)])
def test_thin_transpositions(gpu, thin, batch, big):
    for shape in ((batch, thin, big), (batch, big, thin)):
        x = normal(thin + big, batch * thin * big, 1.0).reshape(shape)
        dx, y = Buffer.from_numpy(x), Buffer(x.nbytes)
        check(hip().shdw_hip_permute(3, ints(list(shape)), ints([0, 2, 1]), dx.ptr, y.ptr, None))
        check(hip().shdw_hip_stream_sync(None))
        got = y.download(count=x.size).reshape(shape[0], shape[2], shape[1])
        assert np.array_equal(got, x.transpose(0, 2, 1)), "%s" % (shape,)
