"""Meshes with vertices of so many cells that no tile of the wanted size can hold
their neighbours (1023 slots), faces (two for each of 512 threads) or both: the
solver takes smaller tiles, and the CSR-gather kernels where none fits.  Runs
against the oracle, 1e-12 in conserved variables; settings that are wrong by
themselves stay refused."""
import numpy as np
import pytest

import tensum_amd as T
import oracle_binding as O
from cases import conserved, rel_l2
from test_gpu_parity import _fan_mesh
from test_stage_gpu import _hub_mesh, _wave

pytestmark = pytest.mark.gpu


def _two_hubs(n):
    """A disk of 2n triangles around two neighbouring inner vertices, each joined
    to one half of the circle, and the two triangles between the halves."""
    t = 2 * np.pi * np.arange(2 * n) / (2 * n)
    x = np.concatenate([[0.3, 0.3], np.cos(t)])
    y = np.concatenate([[0.31, 0.29], np.sin(t)])
    p = lambda k: 2 + k % (2 * n)
    cells = [(0, p(k), p(k + 1)) for k in range(n)] + [(1, p(k), p(k + 1)) for k in range(n, 2 * n)]
    cells += [(0, p(n), 1), (1, p(0), 0)]
    bf = [(p(k), p(k + 1)) for k in range(2 * n)]
    return T.Mesh(x=x, y=y, bface_tag=np.full(2 * n, 1, np.int32), bface_v=np.array(bf, np.int32).ravel(),
                  cell_v=np.array(cells, np.int32).ravel(), periodic_ptr=np.zeros(0, np.int32),
                  periodic_v=np.zeros(0, np.int32), bc={1: ("outlet",)})


# mesh, tile size asked for, tile size in use for Euler (0: the CSR kernels).  The
# viscous cells beside the 800 neighbours of two_hubs_400 (128 + 48 bytes each) are
# more than LDS at any tile size.
MESHES = {"hub_1100": (lambda: _fan_mesh(1100), 0, 0), "two_hubs_505": (lambda: _two_hubs(505), 0, 0),
          "two_hubs_700": (lambda: _two_hubs(700), 0, 0), "two_hubs_400": (lambda: _two_hubs(400), 256, 128)}


@pytest.mark.parametrize("pre", ["auto", "host"])
@pytest.mark.parametrize("model,flux", [("euler", "kepes_tecno_rusanov"), ("ns", "kepes_tecno_roe")])
@pytest.mark.parametrize("kind", sorted(MESHES))
def test_tiles_shrink_or_give_way(kind, model, flux, pre):
    print(kind, model, flux, pre, flush=True)
    make, want, tile = MESHES[kind]
    m = make()
    w = _wave(m)
    prm = T.Params(flux=flux, reconstruct="minmod", cfl=0.3, final_time=1.0, model=model,
                   mu_ref=1e-3 if model == "ns" else 0.0, preprocess=pre, tile_vertices=want)
    s, o = T.Solver(m, prm), O.Oracle(m, prm)
    assert s.tile_vertices == (tile if model == "euler" else 0)
    s.set_state(w)
    o.set_state(w)
    assert s.run(5)[0] == o.run(5)
    assert rel_l2(conserved(s.get_state()), conserved(o.get_state())) <= 1e-12


@pytest.mark.parametrize("kind", ["hub_1100", "plain"])
def test_wrong_settings_stay_refused(kind):
    m = _fan_mesh(1100) if kind == "hub_1100" else _fan_mesh(12)
    base = dict(flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.3, final_time=1.0)
    for bad in (dict(block_fu=1024), dict(block_fu=520), dict(block_grad=1024),
                dict(tile_vertices=257), dict(graph_steps=-1), dict(graph_steps=5000)):
        with pytest.raises(T.TsmError):
            T.Solver(m, T.Params(**base, **bad))


def _with_set(m, vertices):
    """The mesh with the given vertices as one periodic set."""
    v = np.asarray(vertices, np.int32)
    return T.Mesh(**{**m.__dict__, "periodic_ptr": np.array([0, v.size], np.int32), "periodic_v": v})


@pytest.mark.parametrize("size,tile", [(28, 112), (29, 128), (32, 128), (33, None)])
def test_large_periodic_sets(size, tile):
    """A quarter tile has to hold a set: 32 vertices by default, in every scheme."""
    m = T.jittered_mesh(49, seed=2, bc={t: ("outlet",) for t in (1, 2, 3, 4)})
    inner = np.flatnonzero((np.abs(m.x - m.x.mean()) < 0.4 * np.ptp(m.x))
                           & (np.abs(m.y - m.y.mean()) < 0.4 * np.ptp(m.y)))
    m = _with_set(m, inner[::inner.size // size][:size])
    prm = T.Params(model="ns", flux="kepes_tecno_roe", reconstruct="minmod", cfl=0.3, final_time=1.0,
                   mu_ref=1e-3)
    if tile is None:
        with pytest.raises(T.TsmError, match="periodic set larger"):
            T.Solver(m, prm)
        return
    s, o = T.Solver(m, prm), O.Oracle(m, prm)
    assert s.tile_vertices == tile
    w = _wave(m)
    w[m.periodic_v] = w[m.periodic_v[0]]
    s.set_state(w)
    o.set_state(w)
    assert s.run(5)[0] == o.run(5)
    assert rel_l2(conserved(s.get_state()), conserved(o.get_state())) <= 1e-12


def test_smaller_tiles_that_cannot_hold_a_periodic_set_give_way():
    """480 cells around a vertex and six times as many behind them: two rings fit
    LDS at no tile size that still holds a set of eight."""
    m = _hub_mesh(480, 6)
    m = _with_set(m, 500 + 300 * np.arange(8))
    prm = T.Params(flux="kepes_tecno_rusanov", reconstruct="minmod", cfl=0.3, final_time=1.0,
                   tile_vertices=32)
    s = T.Solver(m, prm)
    assert s.tile_vertices in (0, 32)
    s.set_state(_wave(m))
    assert s.run(2)[0] == 2
