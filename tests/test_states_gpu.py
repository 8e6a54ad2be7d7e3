"""States in and out of the device in the caller's vertex order, the vertex that a
refused state is refused for, and groups of contexts that finish at different steps."""
import numpy as np
import pytest

import tensum_amd as T
from cases import vortex, vortex_mesh

pytestmark = pytest.mark.gpu
BASE = dict(flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.8)


@pytest.mark.parametrize("path", ["auto", "csr"])
@pytest.mark.parametrize("n", [3, 16, 33])
def test_states_come_back_as_given(n, path):
    m = vortex_mesh(n)
    s = T.Solver(m, T.Params(**BASE, final_time=1.0, kernel_path=path), n_samples=3)
    w = [vortex(m.x, m.y) * (1 + 0.01 * k) + 1e-3 * np.arange(m.n_vertex)[:, None] for k in range(3)]
    for k in (2, 0, 1):
        s.set_state(w[k], k)
    assert all(np.array_equal(s.get_state(k), w[k]) for k in range(3))
    s.run(3)
    mid = [s.get_state(k) for k in range(3)]
    s.set_state(w[1], 1)
    assert np.array_equal(s.get_state(0), mid[0]) and np.array_equal(s.get_state(2), mid[2])
    assert np.array_equal(s.get_state(1), w[1]) and s.status(1)["iter"] == 0


@pytest.mark.parametrize("comp,value,word", [(0, 0.0, "temperature"), (3, np.nan, "temperature"),
                                             (3, np.inf, "temperature"), (1, np.nan, "velocity"),
                                             (2, -np.inf, "velocity")])
def test_a_refused_state_names_its_first_bad_vertex(comp, value, word):
    m = vortex_mesh(33)
    s = T.Solver(m, T.Params(**BASE, final_time=1.0))
    good = vortex(m.x, m.y)
    s.set_state(good)
    bad = good.copy()
    first = m.n_vertex - 300
    bad[first, comp] = value
    bad[first + 1:, 0] = -1.0
    with pytest.raises(T.TsmError, match=rf"{word}.*vertex {first}\)"):
        s.set_state(bad)
    assert np.array_equal(s.get_state(), good)


@pytest.mark.parametrize("steps", [1, 15, 16, 17, 40, 200])
def test_groups_that_finish_apart(steps):
    """A context takes no launches any more once its samples are done; counts and
    states are those of separate runs."""
    ends = (0.05, 0.4, 1e9)
    out = []
    for grouped in (False, True):
        ss = []
        for k, t in enumerate(ends):
            m = vortex_mesh(17 + 8 * k)
            s = T.Solver(m, T.Params(**BASE, final_time=t), n_samples=2)
            for j in range(2):
                s.set_state(vortex(m.x, m.y), j)
            ss.append(s)
        done = [T.run_group(ss, steps) if grouped else
                np.array([int(np.sum(s.run(steps))) for s in ss]) for _ in range(3)]
        out.append((done, [s.get_state(j) for s in ss for j in range(2)]))
    assert all(np.array_equal(a, b) for a, b in zip(out[0][0], out[1][0]))
    assert all(np.array_equal(a, b) for a, b in zip(out[0][1], out[1][1]))
