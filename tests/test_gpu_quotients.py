"""Quotients by a divisor that many dividends share (quotients, device_common.h): dividends whose
quotient lies as near to the middle between two floats as any, subnormal and zero quotients and
special values, bit for bit against a division; and the rows of the norms that take new forms."""
from fractions import Fraction

import numpy as np
import pytest

from tests import gpuops
from tests.helpers import normal, uniform
from tests.test_gpu_gate import Case

F = np.float32


def odd_mantissa(d):
    b = int(np.frexp(np.float64(d))[0] * (1 << 24))
    while b % 2 == 0:
        b //= 2
    return b


def nearest_dividends(d):
    """Whole numbers a below 2^24 with |a 2^k - M B| = 1 for the mantissa B of d as an odd number and a midpoint M of
    25 bits: a / d is then 1 / 2 B of a last place off the middle between two floats, and no quotient by d that
    is off at all is nearer.  M is the inverse of B or of -B modulo 2^k; of those two modulo 2^25 one has 25 bits."""
    b, near = odd_mantissa(d), []
    for k in (24, 25):
        for sign in (1, -1):
            m = sign * pow(b, -1, 1 << k) % (1 << k)
            m += (1 << 24) if k == 24 else 0
            a = (m * b - sign) >> k
            if m >= 1 << 24 and 0 < a < 1 << 24:
                near.append(a)
    return near


def near_midpoints(d, rng, n):
    """n dividends, the nearest ones and up to three last places beside them, over many powers of two."""
    near = [F(a) for a in nearest_dividends(d)]
    steps = rng.integers(-3, 4, n).astype(np.int32)
    got = np.array([near[k % len(near)] for k in range(n)], F)
    got = np.where(steps == 0, got, (got.view(np.int32) + steps).astype(np.int32).view(F))
    return np.ldexp(got, rng.integers(-20, 3, n) - 24).astype(F)


def gate_case(shape, fill):
    case = Case(shape, None, scale=False, bias=False, relu=False)
    var = case.stats[1]
    d = np.sqrt(np.abs(var * F(0.5)) + F(1e-3))
    case.stats = (np.zeros_like(var), var)
    rng = np.random.default_rng(5)
    x = case.x.reshape(shape[0], shape[1], -1)
    for c in range(shape[1]):
        x[:, c] = fill(d[c], rng, x[:, c].size).reshape(x[:, c].shape)
    case.x = x.reshape(shape)
    return case


def off_the_middle(x, d):
    """How far x / d is from the nearest middle between two floats, in last places of the quotient, exactly."""
    q = abs(Fraction(float(x)) / Fraction(float(d)))
    ulp = Fraction(float(np.spacing(F(float(q)))))
    return abs(q / ulp - q // ulp - Fraction(1, 2))


def test_near_midpoints_are_that_near():
    """The oracle's side: every divisor has such dividends, they are as near as said, and they are among those used."""
    rng = np.random.default_rng(1)
    for d in np.concatenate([uniform(3, 200, 0.3, 3.0), np.array([3, 5, 1.5, 0.75, 16777215], F)]):
        near = nearest_dividends(d)
        assert near
        for a in near:
            assert off_the_middle(F(a), d) == Fraction(1, 2 * odd_mantissa(d))
        x = near_midpoints(d, rng, 64)
        assert np.all(np.isfinite(x)) and min(off_the_middle(v, d) for v in x) == Fraction(1, 2 * odd_mantissa(d))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(9, 64, 28, 28), (9, 64, 9, 9), (3, 40, 45, 45)])
def test_quotients_next_to_midpoints(gpu, shape):
    gate_case(shape, near_midpoints).check(gpu, "midpoints %s" % (shape,))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(9, 64, 28, 28), (9, 64, 9, 9), (3, 40, 45, 45)])
def test_subnormal_zero_and_special_quotients(gpu, shape):
    def fill(d, rng, n):
        v = (np.ldexp(rng.standard_normal(n), rng.integers(-150, -110, n))).astype(F)
        v[rng.random(n) < 0.2] = F(0)
        v[rng.random(n) < 0.1] = F(-0.0)
        v[0] = F(np.float64(d) * 3 * 2.0 ** -150)  # the quotient's own middle, if d leaves it there
        return v
    gate_case(shape, fill).check(gpu, "subnormal %s" % (shape,))
    case = gate_case(shape, fill)
    flat = case.x.reshape(shape[0] * shape[1], -1)
    flat[::3, 1], flat[1::3, 2], flat[2::3, 0] = F(np.inf), F(-np.inf), F(np.nan)
    case.check(gpu, "special %s" % (shape,))


# one to eight vectors on eight lanes, rows in whole lines and not; a wave a row beside 256 lanes
ROWS = [(1027, n) for n in (4, 8, 12, 16, 20, 32, 36, 48, 64, 96, 128, 160, 196, 224, 252, 256)] + \
       [(2049, n) for n in (3072, 3076, 3136, 3840, 3844)] + \
       [(rows, n) for rows in (1023, 1024, 1300) for n in (4100, 5120, 6004, 8188, 8192)] + \
       [(rows, n) for rows in (2048, 2559, 2560, 3277, 4095, 4097) for n in (3076, 3136, 3840)]


@pytest.mark.gpu
@pytest.mark.parametrize("outer,inner", ROWS)
def test_norm_rows_at_the_edges_of_their_forms(gpu, outer, inner):
    x = normal(90, outer * inner, 2.0) + F(0.5)
    s, b = uniform(91, max(inner, outer), 0.5, 1.5), normal(92, max(inner, outer), 0.2)
    rows = x.reshape(outer, inner)
    mean = (rows.astype(np.float64) * np.float64(F(1) / F(inner))).sum(1)
    centred = rows - mean.astype(F)[:, None]
    var = (centred.astype(np.float64) ** 2).sum(1) * np.float64(F(1) / F(inner))
    want = centred / np.sqrt(var + 1e-5)[:, None]
    for kw, w in (({}, want), (dict(scale=s[:inner], bias=b[:inner], scale_num=inner, scale_inner=1), want * s[:inner] + b[:inner]),
                  (dict(scale=s[:outer], bias=b[:outer], scale_num=outer, scale_inner=inner), want * s[:outer, None] + b[:outer, None])):
        got = gpuops.group_norm(x, outer, inner, 1e-5, **kw)
        # eight roundings of a value of order 1, and the affine sum may cancel
        assert np.max(np.abs(got.reshape(outer, inner) - w) / np.maximum(1.0, np.abs(w))) < 8 * 2.0 ** -24
