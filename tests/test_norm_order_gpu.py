"""A sample's logged residuals do not depend on how many samples share its
context.  A step's norm is summed from its tiles' partials by the last stage's own
last wave or by a launch of its own, depending on the tiles of all samples
together; both take the partials in one order, which follows from the mesh's
tiles alone."""
import numpy as np
import pytest

import tensum_amd as T

pytestmark = pytest.mark.gpu


def _wave(m, k):
    w = np.tile(np.array([1.0, 0.2 + 0.1 * k, 0.1, 1.0]), (m.n_vertex, 1))
    w[:, 0] *= 1 + 0.05 * np.sin(2 * m.y + k)
    w[:, 3] *= 1 + 0.05 * np.cos(3 * m.x) * (1 + m.y)
    return w


# 49^2: 151 tiles of 16 vertices, 76 of 32, 601 of 4 (never ended by the last stage)
@pytest.mark.parametrize("tile,counts", [(16, (1, 3, 4, 9)), (32, (1, 6, 7, 20)), (4, (1, 2))])
@pytest.mark.parametrize("how", ["run", "step", "packed"])
def test_a_samples_norms_do_not_depend_on_its_company(tile, counts, how):
    m = T.jittered_mesh(49, seed=2, bc={t: ("outlet",) for t in (1, 2, 3, 4)})
    prm = T.Params(flux="kepes_tecno_rusanov", reconstruct="minmod", cfl=0.4, final_time=10.0,
                   tile_vertices=tile)
    ref = None
    for n in counts:
        print(tile, n, how, flush=True)
        s = T.Solver(m, prm, n_samples=n)
        for k in range(n):
            s.set_state(_wave(m, k), k)
        if how == "run":
            _, log = s.run(8, want_log=True)
            got = np.asarray(log).reshape(n, 8, 4)[0]
        elif how == "step":
            got = np.array([s.step()[1][0] for _ in range(8)])
        else:
            T.run_packed([s], 8)
            got = np.array([s.status(0)["res"], *s.time(0)])
        if ref is None:
            ref = got.copy()
        assert np.array_equal(got, ref), n
