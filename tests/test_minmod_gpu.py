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
    rng = np.random.default_rng(7)
    v = np.concatenate([rng.standard_normal(40), 10.0 ** rng.uniform(-300, 300, 20),
                        -10.0 ** rng.uniform(-300, 300, 20),
                        [0.0, -0.0, np.inf, -np.inf, np.nan, 1.7976931348623157e308, -5e-324, 5e-324]])
    a, b = (x.ravel() for x in np.meshgrid(v, v))
    keep = ~np.isnan(b)  # with the jump itself NaN the flux is NaN whatever the slope
    a, b = a[keep], b[keep]
    with np.errstate(over="ignore"):
        want = _minmod(a, b) + _minmod(b, b)
    got = T.check_math(a, b)[:, 5]
    bad = ~((got == want) | (np.isnan(got) & np.isnan(want)))
    assert not bad.any(), list(zip(a[bad], b[bad], got[bad], want[bad]))[:10]
