"""Evaluations in every form the row count chooses: one or two row tiles a block
(two from 32,768 rows) and more than one chunk of staged rows (64 MiB), the last
one short.  A row's outputs depend on its own inputs alone, so each form gives the
bits of the rows evaluated a few thousand at a time, which are compared with the
FP64 oracle (tolerance as in test_surrogate_gpu.py)."""
import numpy as np
import pytest

import mlp_oracle as MO
from tensum_amd.surrogate import MLP

pytestmark = pytest.mark.gpu

# widths, rows, FP64 moments around the net: two tiles a block; the same in two
# chunks of 233,016 rows; one tile a block in chunks of 32,388 and of 16,194
CASES = [([6, 256, 256, 256, 66], 40001, False), ([6, 256, 256, 256, 66], 40001, True),
         ([5, 200, 33, 7], 65536 + 17, False), ([6, 64, 66], 250007, False),
         ([6, 64, 512], 40000, False), ([6, 64, 512], 17000, True)]


@pytest.mark.parametrize("widths,n,affine", CASES)
def test_rows_do_not_depend_on_how_many_there_are(widths, n, affine):
    print(widths, n, affine, flush=True)
    rng = np.random.default_rng(8)
    net = MLP(widths, max_batch=64, seed=6)
    x = rng.standard_normal((n, widths[0]))
    if affine:
        mom = [rng.random(widths[0]), 0.5 + rng.random(widths[0]),
               rng.standard_normal(widths[-1]), 0.5 + rng.random(widths[-1])]
        call = lambda a: net.affine(a, *mom)
    else:
        x = x.astype(np.float32)
        call = net
    y = call(x)
    step = 4096
    for r in range(0, n, step):
        assert np.array_equal(call(x[r:r + step]), y[r:r + step]), r
    pick = np.concatenate([np.arange(40), rng.integers(0, n, 40), np.arange(n - 40, n)])
    u = x[pick].astype(np.float64)
    if affine:
        u = ((u - mom[0]) / mom[1]).astype(np.float32).astype(np.float64)
    ref, _ = MO.forward(net.params.astype(np.float64), widths, u, bf=True)
    got = y[pick]
    if affine:
        got = (got - mom[2]) / mom[3]
    assert np.linalg.norm(got - ref) <= 5e-3 * np.linalg.norm(ref)
