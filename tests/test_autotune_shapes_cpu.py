"""Autotuner host logic (no GPU, a solver that only answers): no two default shapes
are the same launches, and a tile size that the context does not take is not
timed under its name."""
from types import SimpleNamespace

import pytest

import tensum_amd as T
from tensum_amd import autotune as AT


def _solver(largest, timed):
    """Solvers that halve tiles of more than `largest` vertices, as tsm_create does."""
    class S:
        def __init__(self, mesh, params, n_samples=1):
            tb = params.tile_vertices or 128
            if params.kernel_path == "csr" or params.bc_scheme == "strong":
                tb = 0
            while tb > largest:
                tb //= 2
            self.tile_vertices = tb if tb >= 16 else 0
            self.us = 1000.0 / (self.tile_vertices or 1)

        def set_state(self, w, k): pass
        def run(self, n): pass
        def close(self): pass

        def bench(self, n):
            timed.append(self.tile_vertices)
            return {"step_us": self.us}
    return S


def test_default_shapes_are_different_launches():
    seen = [(c["tile_vertices"], c["block_fu"]) for c in AT.candidates()]
    assert len(seen) == len(set(seen))


@pytest.mark.parametrize("largest", [256, 100])
def test_sizes_that_are_not_taken_are_not_timed(monkeypatch, largest):
    timed = []
    monkeypatch.setattr(AT, "Solver", _solver(largest, timed))
    best, table = AT.autotune(SimpleNamespace(), T.Params(), None)
    assert [sh["tile_vertices"] for sh, _ in table] == timed
    assert max(timed) == best.tile_vertices <= largest


def test_no_size_fits(monkeypatch):
    monkeypatch.setattr(AT, "Solver", _solver(8, []))
    with pytest.raises(T.TsmError, match="no launch shape fits"):
        AT.autotune(SimpleNamespace(), T.Params(), None)


@pytest.mark.parametrize("kw", [dict(kernel_path="csr"), dict(bc_scheme="strong")])
def test_contexts_without_tiles_take_any_shape(monkeypatch, kw):
    timed = []
    monkeypatch.setattr(AT, "Solver", _solver(256, timed))
    _, table = AT.autotune(SimpleNamespace(), T.Params(**kw), None)
    assert len(table) == len(AT.candidates()) and set(timed) == {0}
