"""The minmod slope of the TeCNO flux against the reference's branches
(src/limiter.h): the smaller of two numbers of one sign, zero otherwise, and so
zero where either is NaN: a gradient that has blown up beside finite states
gives the flux no slope at all."""
import numpy as np
import pytest

import tensum_amd as T

pytestmark = pytest.mark.gpu


def _minmod(a, b):
    with np.errstate(invalid="ignore"):
        neg, pos = (a < 0) & (b < 0), (a > 0) & (b > 0)
        return np.where(neg, np.maximum(a, b), np.where(pos, np.minimum(a, b), 0.0))


def test_minmod_takes_the_branches_values():
    """(minmod(2a - b, b) + minmod(b, b)) / 2 for gradients a and jumps b: multiples of
    2^-20, so that 2a - b is exact, and values whose slope is decided by size."""
    rng = np.random.default_rng(7)
    u = rng.integers(-2 ** 22, 2 ** 22, 300) * 2.0 ** -20
    big = np.concatenate([s * 10.0 ** rng.uniform(-300, 300, 20) for s in (1, -1)])
    v = np.concatenate([u, [0.0, -0.0, np.inf, -np.inf, np.nan]])
    a, b = (x.ravel() for x in np.meshgrid(v, u))
    a2, b2 = (x.ravel() for x in np.meshgrid(np.concatenate([big, [0.0, np.inf, -np.inf, np.nan, 5e-324]]),
                                             np.concatenate([big, [0.0, 5e-324, -5e-324]])))
    far = ~((np.abs(a2) > 1e-3 * np.abs(b2)) & (np.abs(a2) < 1e3 * np.abs(b2)))
    a, b = np.concatenate([a, a2[far]]), np.concatenate([b, b2[far]])
    with np.errstate(invalid="ignore", over="ignore"):
        want = 0.5 * (_minmod(2 * a - b, b) + _minmod(b, b))
    got = T.check_math(a, b)[:, 5]
    bad = got != want
    assert not bad.any(), list(zip(a[bad], b[bad], got[bad], want[bad]))[:10]
