"""States in and out on both sides of the size up to which they go through pinned
host memory (16,384 vertices) instead of a copy: 128^2 and 129^2 vertices, several
samples, tiled and CSR, before and between steps; refused states change nothing."""
import numpy as np
import pytest

import tensum_amd as T
from cases import riemann_mesh

pytestmark = pytest.mark.gpu


def _state(m, k):
    w = np.tile(np.array([1.0, 0.2 + 0.1 * k, 0.1, 1.0]), (m.n_vertex, 1))
    w[:, 0] *= 1 + 0.05 * np.sin(2 * m.y + k)
    w[:, 3] += 1e-5 * np.arange(m.n_vertex)
    return w


@pytest.mark.parametrize("kw", [{}, dict(kernel_path="csr"), dict(bc_scheme="strong")])
@pytest.mark.parametrize("n", [3, 45, 128, 129])
def test_states_in_and_out(n, kw):
    m = riemann_mesh(n)
    prm = T.Params(flux="kepes_tecno_rusanov", reconstruct="minmod", cfl=0.4, final_time=10.0, **kw)
    s, one = T.Solver(m, prm, n_samples=3), T.Solver(m, prm)
    for k in (1, 2, 0):
        s.set_state(_state(m, k), k)
    assert all(np.array_equal(s.get_state(k), _state(m, k)) for k in range(3))
    s.run(3)
    mid = [s.get_state(k) for k in range(3)]
    for comp, vertex in ((0, m.n_vertex - 1), (3, 0), (1, m.n_vertex // 2)):
        bad = _state(m, 1)
        bad[vertex, comp] = np.nan
        with pytest.raises(T.TsmError, match=rf"vertex {vertex}\)"):
            s.set_state(bad, 1)
    assert all(np.array_equal(s.get_state(k), mid[k]) for k in range(3))
    s.run(4)
    for k in range(3):
        one.set_state(_state(m, k))
        one.run(7)
        assert np.array_equal(s.get_state(k), one.get_state())
