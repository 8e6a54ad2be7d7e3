"""The stage kernel at the edges of its tables, against the oracle: vertices
with more neighbours than the first chain's eight and a group's seven, vertices
whose two halo rings do not fit LDS at the wanted tile size (smaller tiles are
taken), boundary terms beside them, every tile size from the smallest to the
largest, and runs cut into several calls (the entropy variable kept beside the
state starts anew with each call).  Tolerances as elsewhere: short runs to
1e-12 in conserved variables; runs of one scheme that only differ in their
launch shape are equal to the bit."""
import numpy as np
import pytest

import tensum_amd as T
import oracle_binding as O
from cases import conserved, rel_l2, vortex, vortex_mesh
from test_gpu_parity import _fan_mesh

pytestmark = pytest.mark.gpu


def _hub_mesh(n, s):
    """_fan_mesh's half disk with s outer vertices for every inner one: the
    second halo ring of the centre's tile grows with s while the first does not."""
    th, to = np.pi * np.arange(n + 1) / n, np.pi * np.arange(s * n + 1) / (s * n)
    x = np.concatenate([[0.0], 0.5 * np.cos(th), np.cos(to)])
    y = np.concatenate([[0.0], 0.5 * np.sin(th), np.sin(to)])
    inn, out = 1 + np.arange(n + 1), n + 2 + np.arange(s * n + 1)
    cells = [(0, inn[k], inn[k + 1]) for k in range(n)]
    for k in range(n):
        cells += [(inn[k], out[s * k + j], out[s * k + j + 1]) for j in range(s)]
        cells += [(inn[k], out[s * (k + 1)], inn[k + 1])]
    bf = [(out[-1], inn[n], 1), (inn[n], 0, 1), (0, inn[0], 1), (inn[0], out[0], 1)]
    bf += [(out[k], out[k + 1], 2) for k in range(s * n)]
    return T.Mesh(x=x, y=y, bface_tag=np.array([t for _, _, t in bf], np.int32),
                  bface_v=np.array([[a, b] for a, b, _ in bf], np.int32).ravel(),
                  cell_v=np.array(cells, np.int32).ravel(),
                  periodic_ptr=np.zeros(0, np.int32), periodic_v=np.zeros(0, np.int32),
                  bc={1: ("slip",), 2: ("outlet",)})


def _wave(m):
    w = np.tile(np.array([1.0, 0.2, 0.1, 1.0]), (m.n_vertex, 1))
    w[:, 0] *= 1 + 0.05 * np.sin(2 * m.y)
    w[:, 3] *= 1 + 0.05 * np.cos(3 * m.x) * (1 + m.y)
    return w


@pytest.mark.parametrize("model,flux", [("euler", "kepes_tecno_rusanov"), ("euler", "kepec"),
                                        ("ns", "kepes_tecno_roe"), ("ns", "kepec")])
@pytest.mark.parametrize("cells", [3, 7, 8, 9, 15, 16, 17, 40, 300, (480, 1), (480, 3), (480, 6)])
def test_vertices_with_any_number_of_cells(cells, model, flux):
    print(f"fan of {cells}, {model} {flux}", flush=True)
    m = _hub_mesh(*cells) if isinstance(cells, tuple) else _fan_mesh(cells)
    w = _wave(m)
    prm = T.Params(flux=flux, reconstruct="minmod", cfl=0.3, final_time=1.0, model=model,
                   mu_ref=1e-3 if model == "ns" else 0.0,
                   tile_vertices=32 if isinstance(cells, tuple) else 0)
    s, o = T.Solver(m, prm), O.Oracle(m, prm)
    s.set_state(w)
    o.set_state(w)
    assert s.run(5)[0] == o.run(5)
    assert rel_l2(conserved(s.get_state()), conserved(o.get_state())) <= 1e-12


@pytest.mark.parametrize("kind", ["periodic", "walls"])
def test_launch_shapes_and_cut_runs_agree_bitwise(kind):
    if kind == "periodic":
        m = vortex_mesh(37)
        w = vortex(m.x, m.y)
        base = dict(flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.8, final_time=10.0)
    else:
        st = (1.0, 0.3, 0.0, 1.0)
        m = T.jittered_mesh(37, seed=4, bc={1: ("noslip", (1.1, 0.0, 0.0, 1.0)), 2: ("pressure", st),
                                            3: ("slip",), 4: ("farfield", st)})
        w = np.tile(np.array(st), (m.n_vertex, 1))
        w[:, 0] *= 1 + 0.05 * np.sin(np.pi * m.x)
        base = dict(flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.5, final_time=10.0,
                    model="ns", mu_ref=0.002)
    out = []
    for kw, cuts in (({}, (12,)), ({}, (1, 4, 7)), (dict(tile_vertices=4), (12,)),
                     (dict(tile_vertices=16), (5, 7)), (dict(tile_vertices=100), (12,)),
                     (dict(tile_vertices=256), (12,)), (dict(block_fu=512), (12,)),
                     (dict(preprocess="host"), (12,)), (dict(graph_steps=3), (12,))):
        print(kind, kw, cuts, flush=True)
        s = T.Solver(m, T.Params(**base, **kw))
        s.set_state(w)
        for k in cuts:
            s.run(k)
        out.append(s.get_state())
        assert np.array_equal(out[0], out[-1]), (kw, cuts)


@pytest.mark.parametrize("tile", [4, 5, 6, 16])
def test_steps_end_alike_whoever_ends_them(tile):
    """Contexts of up to 512 tiles end their steps in the last stage, larger ones in
    a launch of its own (2401 vertices, three samples: 1800 tiles or more at 4, 450
    at 16, 57 by default).
    The time steps are minima and equal to the bit; a norm is the root of a sum of
    2401 positive terms taken in another order (2401 eps / 2 = 3e-13 relative)."""
    m = T.jittered_mesh(49, seed=2, bc={t: ("outlet",) for t in (1, 2, 3, 4)})
    base = dict(flux="kepes_tecno_rusanov", reconstruct="minmod", cfl=0.4, final_time=10.0)
    logs = []
    for kw in (dict(), dict(tile_vertices=tile), dict(tile_vertices=tile)):
        s = T.Solver(m, T.Params(**base, **kw), n_samples=3)
        for k in range(3):
            w = _wave(m)
            w[:, 1] += 0.1 * k
            s.set_state(w, k)
        print(tile, kw, T.host_tiling(m, kw.get("tile_vertices", 128))["tiles"], flush=True)
        done, log = s.run(8, want_log=True)
        assert np.all(np.asarray(done) == 8)
        logs.append(np.asarray(log).reshape(3, 8, 4).copy())
    assert np.array_equal(logs[1], logs[2])
    assert np.array_equal(logs[0][..., :3], logs[1][..., :3])
    np.testing.assert_allclose(logs[1][..., 3], logs[0][..., 3], rtol=6e-13, atol=0)
