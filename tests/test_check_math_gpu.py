"""Reciprocal, reciprocal root, root and logarithm of about an ulp
(tensum_amd/csrc/tsm_physics.h) against 80-bit arithmetic on the host.

Bounds.  The hardware estimates are good to 2^-22 at worst; one third-order
step leaves the cube of that.  What remains are roundings, in units of 2^-53
relative: the last multiply-add of the reciprocal, 1; for 1/sqrt(x) also the
rounding of x y in e = 1 - (x y) y, half of whose error is taken into the
result, 1.5; for sqrt(x) the rounding of g = x y, half of which the correction
removes, 1.5.  The logarithm keeps its leading part exactly; its correction
terms are at most 4 per cent of the result and good to 2 ulp, so half an ulp for
the last addition and less than 0.2 more.  Operands: every exponent that the
square of the estimate's step allows; the logarithm over all positive numbers,
subnormal ones included, and the library's value for every other operand."""
import numpy as np
import pytest

import tensum_amd as T

pytestmark = pytest.mark.gpu
LD = np.longdouble
U = LD(2) ** -53


def _operands(lo, hi, n, seed):
    rng = np.random.default_rng(seed)
    e = np.repeat(np.arange(lo, hi + 1), n)
    return np.ldexp(rng.uniform(1.0, 2.0, e.size), e)


@pytest.mark.skipif(np.finfo(LD).nmant < 63, reason="needs 80-bit floating point on the host")
def test_reciprocals_and_roots():
    x = _operands(-500, 500, 1024, 1)
    got = T.check_math(x, np.ones_like(x)).astype(LD)
    X = x.astype(LD)
    for k, (want, bound) in enumerate(((1 / X, 1.0), (1 / np.sqrt(X), 1.5), (np.sqrt(X), 1.5))):
        err = np.max(np.abs(got[:, k] / want - 1)) / U
        print(k, float(err), flush=True)
        assert err <= bound * 1.001
    neg = T.check_math(-x[::64], np.ones(x[::64].size))
    assert np.array_equal(neg[:, 0], -got[::64, 0].astype(np.float64))


@pytest.mark.skipif(np.finfo(LD).nmant < 63, reason="needs 80-bit floating point on the host")
@pytest.mark.parametrize("lo,hi,n", [(-1, 0, 1 << 19), (-1022, 1023, 512), (-40, 40, 1 << 13)])
def test_logarithm(lo, hi, n):
    x = _operands(lo, hi, n, 2)
    got = T.check_math(x, np.ones_like(x))[:, 3]
    want = np.log(x.astype(LD))
    ulp = np.spacing(np.abs(want.astype(np.float64))).astype(LD)
    err = np.max(np.abs(got.astype(LD) - want) / ulp)
    print(lo, hi, float(err), flush=True)
    assert err <= 0.7


def test_logarithm_of_every_kind_of_operand():
    tiny = np.array([5e-324, 1e-323, 3e-310, 2.2250738585072009e-308])
    special = np.array([0.0, -0.0, -1.0, -5e-324, -np.inf, np.inf, np.nan, 1.0])
    got = T.check_math(tiny, np.ones(tiny.size))[:, 3]
    want = np.log(tiny.astype(LD))
    assert np.all(np.abs(got - want) <= 0.7 * np.spacing(np.abs(want.astype(np.float64))))
    out = T.check_math(special, np.ones(special.size))
    assert np.array_equal(out[:, 3], out[:, 4], equal_nan=True)
    assert np.array_equal(out[:, 3], [-np.inf, -np.inf, np.nan, np.nan, np.nan, np.inf, np.nan, 0.0],
                          equal_nan=True)
