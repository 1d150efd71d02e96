"""shdw_hip_squeeze_gate through the C ABI, every form its kernels have: rows whole in LDS and in
chunks, one and several rows a lane, last groups cut short, one to sixteen vectors a lane,
each with rows of whole vectors and not, and with x, another tensor or nothing as the
residual.  Bit for bit against the operators of the oracle; the plane means, 64-bit sums
in another order, to 1e-5.  tests/test_gate_shape_cpu.py checks that the shapes and parts reach the
kernels and forms named here."""
import numpy as np
import pytest

import oracle
import shadow_amd
from shadow_amd import Buffer
from tests.helpers import assert_bit_exact, assert_rel_close, normal, uniform, with_specials
from tests.test_gpu_plane_average import rows_without_signs

pytestmark = pytest.mark.gpu
F = np.float32

FORMS = {
    (516, 1, 84, 84): {"lanes": 256, "turns": 1, "slots": 8, "chunked": True},
    (516, 1, 81, 81): {"lanes": 256, "turns": 1, "slots": 8, "chunked": True},
    (2060, 1, 44, 44): {"lanes": 64, "turns": 1, "slots": 8, "chunked": True},
    (2060, 1, 45, 45): {"lanes": 64, "turns": 1, "slots": 8, "chunked": True},
    (2061, 1, 60, 60): {"lanes": 256, "turns": 2, "slots": 8, "chunked": True, "cut_group": True},
    (2061, 1, 59, 61): {"lanes": 256, "turns": 2, "slots": 8, "chunked": True, "cut_group": True},
    (600, 1, 112, 112): {"lanes": 256, "turns": 1, "slots": 16, "chunked": True},
    (600, 1, 111, 113): {"lanes": 256, "turns": 1, "slots": 16, "chunked": True},
    (3, 2, 112, 112): {"lanes": 256, "turns": 1, "slots": 16, "chunked": False},
    (3, 2, 111, 113): {"lanes": 256, "turns": 1, "slots": 16, "chunked": False},
    (8201, 1, 28, 28): {"lanes": 64, "turns": 2, "slots": 8, "chunked": False, "cut_group": True},
    (8201, 1, 27, 29): {"lanes": 64, "turns": 2, "slots": 8, "chunked": False, "cut_group": True},
    (4101, 1, 31, 33): {"lanes": 64, "turns": 1, "slots": 4, "chunked": False, "cut_group": True},
    (32801, 1, 7, 8): {"lanes": 16, "turns": 2, "slots": 4, "chunked": False, "cut_group": True},
    (32801, 1, 5, 6): {"lanes": 16, "turns": 2, "slots": 4, "chunked": False, "cut_group": True},
    (21867, 3, 2, 2): {"lanes": 16, "turns": 4, "slots": 4, "chunked": False, "cut_group": True},
    (1366, 3, 9, 9): {"lanes": 32, "turns": 1, "slots": 1, "chunked": False, "cut_group": True},
    (5, 3, 9, 9): {"lanes": 256, "turns": 1, "slots": 1, "chunked": False},
    (4099, 1, 1, 3): {"lanes": 16, "turns": 1, "slots": 1, "chunked": False, "cut_group": True},
    (4099, 1, 1, 1): {"lanes": 16, "turns": 1, "slots": 1, "chunked": False, "cut_group": True},
    # a lane a row in the walk, and all lanes together, where a form has both
    (4101, 1, 16, 20): {"lanes": 64, "turns": 1, "slots": 4, "chunked": False, "cut_group": True, "together": False},
    (4101, 1, 17, 17): {"lanes": 64, "turns": 1, "slots": 4, "chunked": False, "cut_group": True, "together": False},
    (4101, 1, 16, 24): {"lanes": 64, "turns": 1, "slots": 4, "chunked": False, "cut_group": True, "together": True},
    (2001, 1, 17, 17): {"lanes": 64, "turns": 1, "slots": 4, "chunked": False, "cut_group": True, "together": True},
    (4101, 1, 13, 13): {"lanes": 64, "turns": 1, "slots": 1, "chunked": False, "cut_group": True, "together": False},
    (2001, 1, 13, 13): {"lanes": 64, "turns": 1, "slots": 1, "chunked": False, "cut_group": True, "together": True},
    (13003, 1, 20, 20): {"lanes": 64, "turns": 3, "slots": 8, "chunked": False, "cut_group": True, "together": False},
    (13003, 1, 19, 19): {"lanes": 64, "turns": 3, "slots": 8, "chunked": False, "cut_group": True, "together": False},
}


# rows of whole vectors behind BatchNorm and ReLU: one to fifteen vectors of 256 lanes a row, the last one whole and
# cut, and 16, 32 and 64 lanes with last groups cut short
WHOLE = [(5, 3, 8, 8), (2, 3, 32, 32), (3, 2, 28, 44), (2, 2, 50, 50), (2, 2, 64, 64), (1, 3, 68, 72), (1, 2, 78, 78), (1, 2, 88, 88),
         (2, 1, 94, 96), (1, 2, 96, 100), (1, 2, 104, 104), (1, 2, 108, 108), (1, 2, 112, 112), (1, 2, 120, 112), (1, 2, 120, 120),
         (1, 2, 120, 128), (32001, 1, 20, 20), (17003, 1, 18, 28), (8201, 1, 28, 28), (4101, 1, 32, 32), (4101, 1, 40, 40), (1025, 1, 56, 56)]


class Case:
    """Inputs of one shape; parts that are left out are None."""

    def __init__(self, shape, residual="other", stats=True, scale=True, bias=True, relu=True, tail_scale=True, tail_bias=True,
                 special=False):
        c = shape[1]
        self.shape, self.relu = shape, relu
        self.x = normal(70, shape, 2.0)
        if special:
            self.x = with_specials(self.x, 3).reshape(shape)
        self.stats = (normal(71, c, 0.3), uniform(72, c, 0.2, 3.0)) if stats else (None, None)
        self.scale = uniform(73, c, 0.5, 1.5) if scale else None
        self.bias = normal(74, c, 0.3) if bias else None
        tail = residual is not None
        self.tail = (uniform(75, c, 0.5, 1.5) if tail and tail_scale else None, normal(76, c, 0.3) if tail and tail_bias else None)
        self.residual = {"x": self.x, "other": normal(77, shape), "first": normal(77, shape), None: None}[residual]
        self.first = residual == "first"

    def want(self):
        shape, c = self.shape, self.shape[1]
        inner = int(np.prod(shape[2:]))
        with np.errstate(all="ignore"):
            f = self.x
            if self.stats[0] is not None:
                f = oracle.batch_norm(f.ravel(), *self.stats, c, inner, F(0.5), F(1e-3)).reshape(shape)
            if self.scale is not None or self.bias is not None:
                f = oracle.scale_bias(f.ravel(), self.scale, self.bias, c, inner).reshape(shape)
            if self.relu:
                f = oracle.activate_op(f, 1)
            y = oracle.binary_op(f, oracle.activate_op(oracle.pooling_op(f, 1, global_pooling=True), 3), operation=2)
            if self.residual is None:
                return y, None
            t = oracle.scale_bias(y.ravel(), *self.tail, c, inner).reshape(shape)
            y = oracle.activate_op(oracle.eltwise_op([self.residual, t] if self.first else [t, self.residual], 1), 1)
            return y, oracle.reduce_op(y, 4, list(range(2, len(shape))))

    def run(self, lib, alias=None, off=(0, 0, 0), mean=True):
        """alias: 'x' or 'residual', which y then is; off: floats that x, the residual and y are off the vector boundary."""
        def buffer(a, at=0):
            if a is None:
                return None
            b = Buffer(4 * (a.size + 4))
            b.upload(np.ascontiguousarray(a, F).ravel(), 4 * at)
            kept.append(b)
            return b.ptr + 4 * at

        kept, n, c = [], self.x.size, self.shape[1]
        x = buffer(self.x, off[0])
        res = x if self.residual is self.x else buffer(self.residual, off[1])
        y_buf = Buffer(4 * (n + 4))
        y = {"x": x, "residual": res, None: y_buf.ptr + 4 * off[2]}[alias]
        m_buf = Buffer(4 * (n // int(np.prod(self.shape[2:])))) if self.residual is not None and mean else None
        shadow_amd.check(lib.shdw_hip_squeeze_gate(
            n, c, int(np.prod(self.shape[2:])), x, buffer(self.stats[0]), buffer(self.stats[1]), 0.5, 1e-3, buffer(self.scale),
            buffer(self.bias), int(self.relu), buffer(self.tail[0]), buffer(self.tail[1]), res, int(self.first), y,
            m_buf.ptr if m_buf else None, None))
        shadow_amd.check(lib.shdw_hip_stream_sync(None))
        if alias is None:
            got = y_buf.download(count=n, offset_bytes=4 * off[2])
        else:
            where = kept[0] if alias == "x" or self.residual is self.x else kept[1]
            got = where.download(count=n, offset_bytes=4 * (off[0] if where is kept[0] else off[1]))
        return got, None if m_buf is None else m_buf.download(count=m_buf.nbytes // 4)

    def check(self, lib, what, **how):
        (got, mean), (want, want_mean) = self.run(lib, **how), self.want()
        assert_bit_exact(got, want.ravel(), what)
        if mean is not None:
            assert assert_rel_close(mean, want_mean.ravel(), 1e-5, what + " mean") == 0


@pytest.mark.parametrize("residual", ["x", "other", "first", None])
@pytest.mark.parametrize("shape", sorted(FORMS))
def test_every_form(gpu, shape, residual):
    Case(shape, residual).check(gpu, "%s %s" % (shape, residual))


# Whole vectors behind BatchNorm and ReLU, with a residual, may be whole_squeeze_gate_kernel's: with one of these two left out
# they are squeeze_gate_kernel's, in the same forms.
GENERIC = [dict(relu=False), dict(stats=False)]


@pytest.mark.parametrize("residual", ["x", "other", "first"])
@pytest.mark.parametrize("parts", GENERIC)
@pytest.mark.parametrize("shape", sorted(s for s in FORMS if int(np.prod(s[2:])) % 4 == 0))
def test_every_form_of_whole_vectors(gpu, shape, parts, residual):
    Case(shape, residual, **parts).check(gpu, "%s %s %s" % (shape, parts, residual))


@pytest.mark.parametrize("residual", ["x", "other"])
@pytest.mark.parametrize("shape", WHOLE)
def test_whole_rows(gpu, shape, residual):
    """Special values among the elements of small shapes; in place of the residual as well."""
    case = Case(shape, residual, special=shape[0] * shape[1] < 32)
    case.check(gpu, "%s %s" % (shape, residual))
    case.check(gpu, "%s %s in place" % (shape, residual), alias="x" if residual == "x" else "residual", mean=False)


# long rows without ReLU, whose sums have signs, whole and chunked
@pytest.mark.parametrize("shape", [(3, 2, 40, 40), (2, 2, 63, 65), (600, 1, 64, 64), (516, 1, 84, 84), (516, 1, 81, 81)])
def test_long_rows_with_signs(gpu, shape):
    Case(shape, "other", relu=False, special=shape[0] < 9).check(gpu, "%s signs" % (shape,))


# Rows whose sums are taken side by side and pass powers of two in every way: of whole_squeeze_gate_kernel and, without
# BatchNorm or without ReLU, of the other kernel; whole, and in chunks that hand the sum on; whole vectors and not.  A
# variance that makes the divisor 1, a mean of 0 and no scale or bias keep the elements as they are.
@pytest.mark.parametrize("parts", [dict(), dict(stats=False), dict(relu=False)])
@pytest.mark.parametrize("shape", [(39, 1, 32, 32), (39, 1, 31, 33), (39, 1, 45, 45), (39, 1, 84, 84), (516, 1, 84, 84), (516, 1, 81, 81)])
def test_sums_side_by_side(gpu, shape, parts):
    case = Case(shape, "other", scale=False, bias=False, **parts)
    planes, length = shape[0], shape[2] * shape[3]
    case.x = rows_without_signs(length, planes, length).reshape(shape)
    if case.stats[0] is not None:
        case.stats = (np.zeros(1, F), np.full(1, 1.998, F))
        assert np.sqrt(F(1.998) * F(0.5) + F(1e-3)) == F(1)
    case.check(gpu, "%s %s" % (shape, parts))


# whole and chunked, whole vectors and not
ALIASED = [(8201, 1, 28, 28), (8201, 1, 27, 29), (2060, 1, 44, 44), (2060, 1, 45, 45), (600, 1, 111, 113), (5, 3, 9, 9), (4099, 1, 1, 3)]


@pytest.mark.parametrize("alias,residual", [("x", "x"), ("x", "other"), ("residual", "other"), ("residual", "first"), ("x", None)])
@pytest.mark.parametrize("shape", ALIASED)
def test_result_in_place_of_an_operand(gpu, shape, alias, residual):
    for parts in [{}] + (GENERIC[:1] if int(np.prod(shape[2:])) % 4 == 0 else []):
        Case(shape, residual, **parts).check(gpu, "%s y is %s, residual %s %s" % (shape, alias, residual, parts), alias=alias)


@pytest.mark.parametrize("off", [(1, 0, 0), (0, 2, 0), (0, 0, 3), (1, 1, 1)])
@pytest.mark.parametrize("shape", [(8201, 1, 28, 28), (2060, 1, 44, 44), (21867, 3, 2, 2)])
def test_pointers_off_the_vector_boundary(gpu, shape, off):
    Case(shape, "other").check(gpu, "%s off %s" % (shape, off), off=off)


@pytest.mark.parametrize("shape", [(6, 5, 7, 9), (2, 3, 8, 12), (2, 3, 4, 5, 6)])
@pytest.mark.parametrize("parts", [
    dict(stats=False, scale=False, bias=False, relu=False), dict(stats=False, scale=False, bias=False),  # ReLU alone
    dict(scale=False, bias=False), dict(scale=False, bias=False, relu=False),                            # BatchNorm alone
    dict(stats=False, bias=False), dict(stats=False, scale=False), dict(scale=False), dict(bias=False, relu=False)])
@pytest.mark.parametrize("tail", [dict(residual=None), dict(tail_bias=False), dict(tail_scale=False, residual="first")])
def test_parts_left_out(gpu, shape, parts, tail):
    """Fronts and tails of any parts, special values among the elements, volumes as well as planes."""
    Case(shape, special=True, **parts, **{"residual": "other", **tail}).check(gpu, "%s %s %s" % (shape, parts, tail))


def test_no_mean_asked_for(gpu):
    Case((2060, 1, 45, 45), "x").check(gpu, "no mean", mean=False)
