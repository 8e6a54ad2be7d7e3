"""Many contexts at once: the small arrays of a context share allocations of their
own, so contexts beside one another, created and destroyed in any order, give the
results of one alone, and destroying them gives their memory back."""
import numpy as np
import pytest

import tensum_amd as T
from cases import vortex, vortex_mesh

pytestmark = pytest.mark.gpu


def _free():
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("path", ["auto", "csr"])
def test_contexts_beside_one_another(path):
    ms = [vortex_mesh(n) for n in (3, 9, 17, 33)]
    prm = T.Params(flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.8, final_time=10.0,
                   kernel_path=path)
    want = []
    for m in ms:
        s = T.Solver(m, prm)
        s.set_state(vortex(m.x, m.y))
        s.run(9)
        want.append(s.get_state())
        s.close()
    order = np.random.default_rng(1).permutation(4 * 12) % 4
    ss = []
    for i, k in enumerate(order):
        s = T.Solver(ms[k], prm)
        s.set_state(vortex(ms[k].x, ms[k].y))
        s.run(4)
        ss.append((k, s))
        if i % 3 == 2:
            ss.pop(i // 3)[1].close()
    for k, s in ss:
        s.run(5)
        assert np.array_equal(s.get_state(), want[k])


def test_memory_comes_back():
    m = vortex_mesh(65)
    prm = T.Params(flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.8, final_time=10.0)
    T.Solver(m, prm).close()
    before = _free()
    for _ in range(30):
        T.Solver(m, prm, n_samples=2).close()
    assert before - _free() <= 16 << 20  # the runtime's own pools may move by a few MB
