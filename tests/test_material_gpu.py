"""Material constants set between steps: the sample goes on as one of a context that
was created with them, the others are not touched."""
import numpy as np
import pytest

import tensum_amd as T
from cases import vortex, vortex_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["auto", "csr"])
def test_material_set_between_steps(path):
    m = vortex_mesh(17)
    base = dict(flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.5, final_time=1e9, kernel_path=path)
    s = T.Solver(m, T.Params(**base), n_samples=3)
    for k in range(3):
        s.set_state(vortex(m.x, m.y) * (1 + 0.01 * k), k)
    s.run(3)
    mid = [s.get_state(k) for k in range(3)]
    s.set_material(1, 1.3, 0.9)
    with pytest.raises(T.TsmError):
        s.set_material(2, 1.0, 0.9)
    with pytest.raises(T.TsmError):
        s.set_material(2, 1.3, -1.0)
    s.run(4)
    for k, kw in enumerate(({}, dict(gamma=1.3, gas_const=0.9), {})):
        o = T.Solver(m, T.Params(**base, **kw))
        o.set_state(mid[k])
        o.run(4)
        assert np.array_equal(s.get_state(k), o.get_state())


@pytest.mark.parametrize("path", ["auto", "csr"])
def test_queries_after_a_material(path):
    m = vortex_mesh(17)
    base = dict(flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.5, final_time=1e9, kernel_path=path)
    w = vortex(m.x, m.y)
    s, o = T.Solver(m, T.Params(**base)), T.Solver(m, T.Params(**base, gamma=1.3, gas_const=0.9))
    s.set_state(w)
    o.set_state(w)
    s.gradients()  # with the old constants
    s.set_material(0, 1.3, 0.9)
    assert np.array_equal(s.gradients(), o.gradients())
    assert np.array_equal(s.residual(), o.residual())
