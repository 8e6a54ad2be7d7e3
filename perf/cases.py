"""The work this library is used for, as measured cases: whole runs of the
finite-volume solver from the smallest mesh to the largest, batches of Monte
Carlo samples, multilevel batches, a run watched step by step, and the
training and evaluation of the surrogate network.

listed() names the cases, draw() makes more of the same ranges, prepare()
builds what a program holds before the call (mesh, solver context or network,
inputs made from the seed), run() is one pass through the public entry points,
work() the bytes and operations the pass cannot do without, and exact() the
same results by plain numpy in 64 bits: the numerical scheme written out over
edge and cell arrays, without the library's code.
"""
import numpy as np
import torch

import tensum_amd as T
from tensum_amd import uq
from tensum_amd.surrogate import Surrogate

# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
# the solver settings each problem is run with
RUSANOV, ROE, KEPEC = "kepes_tecno_rusanov", "kepes_tecno_roe", "kepec"
WALL_T = 1.1
INFLOW = (1.0, 0.3, 0.0, 1.0)


def listed():
    return [
        # a quick look at a shock problem on a toy mesh: every launch and every
        # host call counts, nothing fills the chip
        _run("shock_33", "riemann", 33, 20, RUSANOV, "minmod"),
        # the convergence-study mesh, one sample, periodic sides
        _run("vortex_129", "vortex", 129, 96, ROE, "minmod"),
        # an odd, ragged middle size, RK4 and an unlimited reconstruction
        _run("vortex_390_rk4", "vortex", 390, 60, RUSANOV, "second", scheme="rk4"),
        # the production run: a shock problem on a million vertices
        _run("shock_1025", "riemann", 1025, 334, RUSANOV, "minmod"),
        # viscous decay on a periodic box, central entropy-conserving flux
        _run("taylor_green_513", "tgv", 513, 200, KEPEC, "first"),
        # viscous flow along walls: boundary conditions of four kinds
        _run("channel_257", "channel", 257, 200, ROE, "minmod"),
        # the driver's loop: one step at a time, its log read after each
        {"name": "watched_257", "kind": "watch", "problem": "riemann", "n": 257, "steps": 40,
         "flux": RUSANOV, "rec": "minmod", "scheme": "ssprk3"},
        # Monte Carlo over uncertain vortices, all samples in one context
        {"name": "batch_vortex_129x64", "kind": "batch", "problem": "vortex", "n": 129,
         "samples": 64, "t_end": 2.0, "rec": "minmod"},
        # the coarse training solves of the shock study (first order, as that study runs)
        {"name": "batch_shock_257x32", "kind": "batch", "problem": "riemann", "n": 257,
         "samples": 32, "t_end": 0.06, "rec": "first"},
        # three levels of a multilevel study advanced together
        {"name": "levels_65_129_257", "kind": "levels", "coarse": 65, "levels": 3,
         "samples": 256, "t_end": 0.8},
        # the surrogate: minibatch training on solver samples ...
        {"name": "fit_2048", "kind": "fit", "rows": 2048, "epochs": 4, "batch": 64, "n_in": 6,
         "hidden": 256, "n_out": 66},
        # ... and the large evaluation that the control variate averages
        {"name": "predict_65536", "kind": "predict", "rows": 65536, "n_in": 6, "hidden": 256,
         "n_out": 66},
    ]


def _run(name, problem, n, steps, flux, rec, scheme="ssprk3"):
    return {"name": name, "kind": "run", "problem": problem, "n": n, "steps": steps, "flux": flux,
            "rec": rec, "scheme": scheme}


def _log_int(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


def draw(rng):
    kind = rng.choice(["run"] * 5 + ["watch", "batch", "batch", "levels", "fit", "predict"])
    if kind in ("run", "watch"):
        problem = rng.choice(["riemann", "vortex", "tgv", "channel"])
        n = _log_int(rng, 25, 1025 if kind == "run" else 400)
        if problem in ("tgv", "channel"):
            n = min(n, 640)
        # never more vertex steps than the production run's
        steps = max(5, min(334, int(rng.uniform(2e5, 1.2e8) / n ** 2)))
        if kind == "watch":
            steps = rng.randint(5, 60)
        scheme = "ssprk3" if problem == "channel" else rng.choice(["ssprk3"] * 3 + ["rk4", "heuns"])
        if problem == "tgv":
            flux, rec = rng.choice([(KEPEC, "first"), (ROE, "minmod")])
        else:
            flux = ROE if problem == "channel" else rng.choice([RUSANOV, ROE])
            rec = rng.choice(["minmod", "minmod", "first"] if problem == "riemann"
                             else ["minmod", "minmod", "second", "first"])
        if problem == "riemann":
            steps = min(steps, 200)
            flux = RUSANOV
        c = _run("", problem, n, steps, flux, rec, scheme)
        del c["name"]
        return dict(c, kind=kind)
    if kind == "batch":
        problem = rng.choice(["vortex", "riemann"])
        n = _log_int(rng, 33, 257)
        samples = max(2, min(512, int(rng.uniform(2e5, 1.0e6) / n ** 2)))
        t_end = rng.uniform(0.2, 1.2) if problem == "vortex" else rng.uniform(0.01, 0.05)
        return {"kind": "batch", "problem": problem, "n": n, "samples": samples,
                "t_end": round(t_end, 4), "rec": "minmod" if problem == "vortex" else "first"}
    if kind == "levels":
        return {"kind": "levels", "coarse": rng.randint(33, 65), "levels": rng.randint(2, 3),
                "samples": rng.randint(16, 200), "t_end": round(rng.uniform(0.1, 0.7), 4)}
    hidden = rng.choice([64, 128, 200, 256])
    if kind == "fit":
        return {"kind": "fit", "rows": _log_int(rng, 100, 2048), "epochs": rng.randint(1, 4),
                "batch": rng.choice([32, 64, 128, 100]), "n_in": rng.randint(3, 8),
                "hidden": hidden, "n_out": rng.randint(10, 80)}
    return {"kind": "predict", "rows": _log_int(rng, 100, 65536), "n_in": rng.randint(3, 8),
            "hidden": hidden, "n_out": rng.randint(10, 80)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _mesh(problem, n, seed):
    seed = seed % 100003
    if problem == "riemann":
        return T.jittered_mesh(n, box=(0.0, 1.0, 0.0, 1.0), jitter=0.2, seed=seed,
                               bc={t: ("outlet",) for t in (1, 2, 3, 4)})
    if problem == "vortex":
        return T.jittered_mesh(n, box=(-5.0, 5.0, -5.0, 5.0), jitter=0.2, seed=seed, periodic=True)
    if problem == "tgv":
        return T.jittered_mesh(n, box=(0.0, 2 * np.pi, 0.0, 2 * np.pi), jitter=0.2, seed=seed,
                               periodic=True)
    return T.jittered_mesh(n, box=(0.0, 1.0, 0.0, 1.0), jitter=0.2, seed=seed,
                           bc={1: ("noslip", (WALL_T, 0.0, 0.0, 1.0)), 2: ("pressure", INFLOW),
                               3: ("slip",), 4: ("farfield", INFLOW)})


def _params(problem, flux, rec, scheme, t_end=None):
    kw = dict(flux=flux, reconstruct=rec, time_scheme=scheme)
    if problem == "riemann":
        return T.Params(cfl=0.5, final_time=t_end or 0.8, **kw)
    if problem == "vortex":
        return T.Params(cfl=0.8, final_time=t_end or 1e9, **kw)
    if problem == "tgv":
        return T.Params(model="ns", cfl=0.5, final_time=1e9, mu_ref=1.0 / 1600.0, prandtl=0.72, **kw)
    return T.Params(model="ns", cfl=0.5, final_time=1e9, mu_ref=0.002, prandtl=0.72, **kw)


def _state(problem, mesh, rng):
    x, y = mesh.x, mesh.y
    if problem == "riemann":
        # the four-quadrant problem with three tenths of its jumps, which the
        # limited second-order scheme carries through some hundred steps
        sx, sy = rng.uniform(0.78, 0.82, 2)
        w = uq.riemann_state(x, y, sx, sy, 1.0, 1.0, 1.0, 1.0)
        rho = 1.5 + 0.3 * (w[:, 3] / w[:, 0] - 1.5)
        p = 1.5 + 0.3 * (w[:, 3] - 1.5)
        return np.stack([p / rho, 0.3 * w[:, 1], 0.3 * w[:, 2], p], 1)
    if problem == "vortex":
        b, xc, yc = rng.uniform(4.0, 6.0), rng.uniform(-0.5, 0.5), rng.uniform(-0.5, 0.5)
        return uq.vortex_state(x, y, b, xc, yc, 1.4, rng.uniform(0.4, 0.6))
    if problem == "tgv":  # Mach 0.1, rho = 1
        a, b = rng.uniform(0, 2 * np.pi, 2)
        p = 1.0 / 0.014 + 0.25 * (np.cos(2 * (x + a)) + np.cos(2 * (y + b)))
        return np.stack([p, np.sin(x + a) * np.cos(y + b), -np.cos(x + a) * np.sin(y + b), p], 1)
    a, b = rng.uniform(0.5, 1.5, 2)
    return np.stack([1.0 + 0.02 * a * np.sin(np.pi * x) * np.cos(np.pi * y),
                     0.3 * (1 - np.exp(-8 * y)) + 0.01 * b * np.sin(2 * np.pi * y),
                     0.01 * np.cos(np.pi * x) * np.sin(np.pi * y),
                     1.0 + 0.01 * a * np.cos(np.pi * (x + b * y))], 1)


def _inputs(problem, samples, seed):
    """Uncertain inputs, uniform in the problem's bounds."""
    u = np.random.default_rng(seed).random((samples, len(problem.bounds)))
    return uq.map_inputs(u, problem.bounds)


def _levels(case):
    """(mesh size, samples) of each level: half the spacing, a quarter of the samples."""
    return [((case["coarse"] - 1) * 2 ** k + 1, max(2, case["samples"] // 4 ** k))
            for k in range(case["levels"])]


def _problem(case):
    if case.get("problem") == "riemann":
        return uq.riemann_problem(final_time=case["t_end"], reconstruct=case["rec"])
    return uq.vortex_problem(final_time=case["t_end"])


def _widths(case):
    return [case["n_in"], case["hidden"], case["hidden"], case["hidden"], case["n_out"]]


def _net_inputs(case, seed):
    rng = np.random.default_rng(seed)
    w = _widths(case)
    p = [q for a, b in zip(w[:-1], w[1:])
         for q in (rng.uniform(-1, 1, (b, a)) * np.sqrt(3.0 / a), 0.1 * rng.standard_normal(b))]
    u = rng.random((case["rows"], case["n_in"]))
    k = np.arange(1, case["n_out"] + 1)[None, :]
    q = (np.sin(np.pi * (u @ np.linspace(0.2, 1.0, case["n_in"]))[:, None] * k / 33.0)
         + u[:, :1] ** 2)
    return u, q, np.concatenate([a.ravel() for a in p]).astype(np.float32)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("run", "watch"):
        m = _mesh(case["problem"], case["n"], seed)
        s = T.Solver(m, _params(case["problem"], case["flux"], case["rec"], case["scheme"]))
        return {"case": case, "solver": s, "w0": _state(case["problem"], m, rng)}
    if kind == "batch":
        p = _problem(case)
        m = _mesh(case["problem"], case["n"], seed)
        return {"case": case, "problem": p, "mesh": m, "inputs": _inputs(p, case["samples"], seed),
                "solver": T.Solver(m, p.params, n_samples=case["samples"])}
    if kind == "levels":
        p = _problem(case)
        st = {"case": case, "problem": p, "mesh": [], "inputs": [], "solver": []}
        for k, (n, ns) in enumerate(_levels(case)):
            m = _mesh("vortex", n, seed + k)
            st["mesh"].append(m)
            st["inputs"].append(_inputs(p, ns, seed + k))
            st["solver"].append(T.Solver(m, p.params, n_samples=ns))
        return st
    u, q, p0 = _net_inputs(case, seed)
    net = Surrogate(case["n_in"], case["n_out"], hidden=(case["hidden"],) * 3, max_batch=4096)
    net.net.params = p0
    if kind == "predict":  # standardisation as a fit leaves it
        net.mu_x, net.sd_x = u.mean(0), u.std(0) + 1e-12
        net.mu_y, net.sd_y = q.mean(0), q.std(0) + 1e-30
    return {"case": case, "net": net, "u": u, "q": q, "p0": p0}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "run":
        s = st["solver"]
        s.set_state(st["w0"])
        done = s.run(case["steps"])
        return {"steps": done, "state": s.get_state()}
    if kind == "watch":
        s = st["solver"]
        s.set_state(st["w0"])
        log = np.zeros((case["steps"], 4))
        bounds = np.zeros((case["steps"], 10))
        for k in range(case["steps"]):
            dt, res = s.step()
            ke, ent = s.global_all()
            log[k] = dt[0], res[0], ke[0], ent[0]
            bounds[k] = s.bounds()
        return {"log": log, "bounds": bounds, "state": s.get_state()}
    if kind == "batch":
        s = uq.make_batch(st["problem"], st["mesh"], st["inputs"], st["solver"])
        uq.advance([s])
        mean, m2, s2 = s.moments()
        return {"qoi": uq.qoi(st["problem"], s), "mean": mean, "m2": m2, "s2": s2}
    if kind == "levels":
        ss = [uq.make_batch(st["problem"], m, i, s)
              for m, i, s in zip(st["mesh"], st["inputs"], st["solver"])]
        uq.advance(ss)
        return {"qoi": [uq.qoi(st["problem"], s) for s in ss], "mean": [s.moments()[0] for s in ss]}
    net = st["net"]
    if kind == "fit":
        # every fit starts from the same weights, in a network that has taken no step
        net.net.close()
        net = st["net"] = Surrogate(case["n_in"], case["n_out"], hidden=(case["hidden"],) * 3,
                                    max_batch=4096)
        net.net.params = st["p0"]
        loss = net.fit(st["u"], st["q"], epochs=case["epochs"], batch=case["batch"], lr=2e-3)
        return {"loss": loss, "params": net.net.params}
    return net(st["u"])


# ---------------------------------------------------------------------------
# bytes and operations
# ---------------------------------------------------------------------------
# FP64 operations of the scheme: one edge flux with limited reconstruction
# (two logarithmic means, three projections, eight minmods), the central flux
# alone, the gradient of one vertex, its update (two logarithms), its viscous terms
OPS = {"tecno": 330, "tecno_first": 200, "kepec": 110, "gradient": 200, "update": 230, "viscous": 900}
STAGES = {"ssprk3": 3, "rk4": 4, "heuns": 2}


def _solver_work(nv, vertex_steps, nst, flux, rec, ns):
    """Each stage reads its input state, the step's first state and the
    geometry (3 edges of normal and end points, position, area) and writes its
    output state, once per vertex."""
    per_stage = 3 * (OPS["kepec"] if flux == KEPEC else
                     OPS["tecno_first"] if rec == "first" else OPS["tecno"]) + OPS["update"]
    if flux != KEPEC and rec != "first":
        per_stage += OPS["gradient"]
    if ns:
        per_stage += OPS["viscous"]
    return {"bytes": vertex_steps * nst * (32 + 32 + 32) + nv * (3 * 24 + 24),
            "flops": vertex_steps * nst * per_stage}


def _steps_to(n, t_end, problem="vortex"):
    """About how many steps the batched problems take."""
    per = 1.17 if problem == "vortex" else 39.0
    return max(1.0, per * t_end * (n - 1))


def work(case):
    kind = case["kind"]
    if kind in ("run", "watch"):
        n2 = case["n"] ** 2
        w = _solver_work(n2, n2 * case["steps"], STAGES[case["scheme"]], case["flux"], case["rec"],
                         case["problem"] in ("tgv", "channel"))
        return {"bytes": w["bytes"] + 64 * n2, "flops": w["flops"]}
    if kind == "batch":
        n2 = case["n"] ** 2
        steps = _steps_to(case["n"], case["t_end"], case["problem"])
        w = _solver_work(n2, n2 * steps * case["samples"], 3,
                         ROE if case["problem"] == "vortex" else RUSANOV, case["rec"], False)
        return {"bytes": w["bytes"] + n2 * (32 * case["samples"] + 120), "flops": w["flops"]}
    if kind == "levels":
        tot = {"bytes": 0.0, "flops": 0.0}
        for n, ns in _levels(case):
            w = _solver_work(n * n, n * n * _steps_to(n, case["t_end"]) * ns, 3, ROE, "minmod", False)
            tot = {"bytes": tot["bytes"] + w["bytes"] + n * n * (32 * ns + 40),
                   "flops": tot["flops"] + w["flops"]}
        return tot
    w = _widths(case)
    macs = sum(a * b for a, b in zip(w[:-1], w[1:]))
    npar = macs + sum(w[1:])
    io = 4 * case["rows"] * (w[0] + w[-1])
    if kind == "fit":
        return {"bytes": io * case["epochs"] + 8 * npar, "flops": 6.0 * macs * case["rows"] * case["epochs"]}
    return {"bytes": io + 4 * npar, "flops": 2.0 * macs * case["rows"]}


# ---------------------------------------------------------------------------
# the same results in 64 bits, by plain numpy
# ---------------------------------------------------------------------------
class _Grid:
    """Median-dual geometry: unique edges with dual normals, outer edges."""

    def __init__(self, m):
        self.x, self.y = m.x, m.y
        nv = self.nv = m.x.size
        c = self.c = m.cell_v.reshape(-1, 3).astype(np.int64)
        X, Y = m.x[c], m.y[c]
        self.X, self.Y = X, Y
        cx, cy = X.sum(1) / 3.0, Y.sum(1) / 3.0
        self.carea = 0.5 * ((X[:, 1] - X[:, 0]) * (Y[:, 2] - Y[:, 0])
                            - (X[:, 2] - X[:, 0]) * (Y[:, 1] - Y[:, 0]))
        a = np.concatenate([c[:, 0], c[:, 1], c[:, 2]])
        b = np.concatenate([c[:, 1], c[:, 2], c[:, 0]])
        tx = np.tile(cx, 3) - 0.5 * (m.x[a] + m.x[b])
        ty = np.tile(cy, 3) - 0.5 * (m.y[a] + m.y[b])
        nx, ny = ty, -tx  # from a to b
        lo, hi = np.minimum(a, b), np.maximum(a, b)
        sg = np.where(a == lo, 1.0, -1.0)
        key, inv = np.unique(lo * nv + hi, return_inverse=True)
        inv = inv.reshape(-1)
        self.l, self.r = key // nv, key % nv
        self.nx = np.bincount(inv, nx * sg, key.size)
        self.ny = np.bincount(inv, ny * sg, key.size)
        self.ar = np.sqrt(self.nx ** 2 + self.ny ** 2)
        self.dx, self.dy = m.x[self.r] - m.x[self.l], m.y[self.r] - m.y[self.l]
        area = np.zeros(nv)
        for j in range(3):
            area += np.bincount(c[:, j], self.carea / 3.0, nv)
        # periodic sets: one number per vertex, the same for a set's members
        self.set_of = None
        self.weight = np.ones(nv)
        if m.periodic_ptr.size:
            g = np.arange(nv)
            for k in range(m.periodic_ptr.size - 1):
                mem = m.periodic_v[m.periodic_ptr[k]:m.periodic_ptr[k + 1]]
                g[mem] = mem[0]
                self.weight[mem] = 1.0 / mem.size
            self.set_of = g
        self.area = self.gather(area)
        # normals of the corners' cell shape functions (twice the area times the gradient)
        self.Nx = np.stack([Y[:, 1] - Y[:, 2], Y[:, 2] - Y[:, 0], Y[:, 0] - Y[:, 1]], 1)
        self.Ny = np.stack([X[:, 2] - X[:, 1], X[:, 0] - X[:, 2], X[:, 1] - X[:, 0]], 1)
        # outer edges that are not periodic
        bv, bt = m.bface_v.reshape(-1, 2).astype(np.int64), m.bface_tag
        keep = np.array([m.bc[int(t)][0] != "periodic" for t in bt], dtype=bool)
        bv, bt = bv[keep], bt[keep]
        self.nb = bt.size
        if not self.nb:
            return
        ce, cj = np.tile(np.arange(c.shape[0]), 3), np.repeat(np.arange(3), c.shape[0])
        order = np.argsort(lo * nv + hi, kind="stable")
        k = np.minimum(bv[:, 0], bv[:, 1]) * nv + np.maximum(bv[:, 0], bv[:, 1])
        at = order[np.searchsorted((lo * nv + hi)[order], k)]
        self.bcell = ce[at]
        self.b0, self.b1 = a[at], b[at]  # counter-clockwise: outward = (dy, -dx)
        self.bnx, self.bny = m.y[self.b1] - m.y[self.b0], m.x[self.b0] - m.x[self.b1]
        e = np.searchsorted(key, k)
        self.hx, self.hy = self.nx[e], self.ny[e]  # half dual face of the outer edge
        self.btype = [m.bc[int(t)][0] for t in bt]
        self.bval = np.array([m.bc[int(t)][1] if len(m.bc[int(t)]) > 1 else (1, 0, 0, 1) for t in bt],
                             dtype=float)
        self.kinds = sorted(set(self.btype))
        self.btype = np.array(self.btype)
        self.wall = np.zeros(c.shape[0], bool)
        self.wall[self.bcell] = True

    def add(self, i, v):
        return np.stack([np.bincount(i, v[:, k], self.nv) for k in range(v.shape[1])], 1)

    def gather(self, v):
        """Sums over the members of each periodic set."""
        if self.set_of is None:
            return v
        if v.ndim == 1:
            return np.bincount(self.set_of, v, self.nv)[self.set_of]
        return self.add(self.set_of, v)[self.set_of]


class _Scheme:
    def __init__(self, mesh, problem, flux, rec, scheme, gam=1.4, t_end=None):
        self.g, self.flux, self.rec, self.scheme, self.gam = _Grid(mesh), flux, rec, scheme, gam
        self.ns = problem in ("tgv", "channel")
        self.cfl = 0.8 if problem == "vortex" else 0.5
        self.mu = 1.0 / 1600.0 if problem == "tgv" else 0.002
        self.pr = 0.72
        self.t_end = t_end

    # pointwise -----------------------------------------------------------
    def ent(self, w):
        rho, beta = w[:, 3] / w[:, 0], 0.5 / w[:, 0]
        s = np.log(w[:, 3]) - self.gam * np.log(rho)
        u, v = w[:, 1], w[:, 2]
        return np.stack([(self.gam - s) / (self.gam - 1) - beta * (u * u + v * v), 2 * beta * u,
                         2 * beta * v, -2 * beta], 1)

    def con(self, w):
        rho = w[:, 3] / w[:, 0]
        return np.stack([rho, rho * w[:, 1], rho * w[:, 2], w[:, 3] / (self.gam - 1)
                         + 0.5 * rho * (w[:, 1] ** 2 + w[:, 2] ** 2)], 1)

    def prim(self, U):
        u, v = U[:, 1] / U[:, 0], U[:, 2] / U[:, 0]
        p = (self.gam - 1) * (U[:, 3] - 0.5 * (U[:, 1] ** 2 + U[:, 2] ** 2) / U[:, 0])
        return np.stack([p / U[:, 0], u, v, p], 1)

    @staticmethod
    def logmean(a, b):
        f = (b - a) / (b + a)
        u = f * f
        near = u < 1e-2
        with np.errstate(divide="ignore", invalid="ignore"):
            far = 0.5 * np.log(b / a) / np.where(near, 1.0, f)
        return 0.5 * (a + b) / np.where(near, 1 + u / 3 + u * u / 5 + u * u * u / 7, far)

    def one_state(self, kind, w, val, nx, ny):
        w = w.copy()
        if kind == "slip":
            vn = (w[:, 1] * nx + w[:, 2] * ny) / (nx * nx + ny * ny)
            w[:, 1] -= vn * nx
            w[:, 2] -= vn * ny
        elif kind == "noslip":
            w[:, :3] = val[:, :3]
        elif kind == "pressure":
            w[:, 3] = val[:, 3]
        return w

    def bstates(self, w, i, nx, ny):
        out = w[i].copy()
        for k in self.g.kinds:
            q = self.g.btype == k
            out[q] = self.one_state(k, w[i[q]], self.g.bval[q], nx[q], ny[q])
        return out

    # operators -----------------------------------------------------------
    def cell_gradients(self, w, V):
        g = self.g
        G = np.zeros((g.c.shape[0], 4, 2))
        for j in range(3):
            G[:, :, 0] += g.Nx[:, j:j + 1] * V[g.c[:, j]]
            G[:, :, 1] += g.Ny[:, j:j + 1] * V[g.c[:, j]]
        if g.nb:
            dq = np.zeros((g.nb, 4))
            for i in (g.b0, g.b1):
                dq += 0.5 * (self.ent(self.bstates(w, i, g.bnx, g.bny)) - V[i])
            np.add.at(G[:, :, 0], g.bcell, g.bnx[:, None] * dq)
            np.add.at(G[:, :, 1], g.bcell, g.bny[:, None] * dq)
        return G

    def edge_flux(self, w, V, dV):
        g = self.g
        d = None
        if dV is not None:  # the end points' gradients along the edge
            d = [dV[i, :, 0] * g.dx[:, None] + dV[i, :, 1] * g.dy[:, None] for i in (g.l, g.r)]
        return self.two_point(w[g.l], w[g.r], V[g.l], V[g.r], d, g.nx, g.ny)

    def two_point(self, wl, wr, Vl, Vr, d, nx, ny):
        """Numerical flux between two states through (nx, ny); d: the
        projected gradients, None without reconstruction."""
        gam = self.gam
        area = np.sqrt(nx * nx + ny * ny)
        ux, uy = nx / area, ny / area
        rl, rr = wl[:, 3] / wl[:, 0], wr[:, 3] / wr[:, 0]
        bl, br = 0.5 / wl[:, 0], 0.5 / wr[:, 0]
        rho, beta = self.logmean(rl, rr), self.logmean(bl, br)
        p = 0.5 * (rl + rr) / (bl + br)
        vx, vy = 0.5 * (wl[:, 1] + wr[:, 1]), 0.5 * (wl[:, 2] + wr[:, 2])
        vn = vx * ux + vy * uy
        q2 = 0.5 * (wl[:, 1] ** 2 + wl[:, 2] ** 2 + wr[:, 1] ** 2 + wr[:, 2] ** 2)
        m = rho * vn
        fx, fy = ux * p + vx * m, uy * p + vy * m
        e = 0.5 * (1 / ((gam - 1) * beta) - q2) * m + fx * vx + fy * vy
        F = np.stack([m, fx, fy, e], 1)
        if self.flux == KEPEC:
            return F * area[:, None]
        a = np.sqrt(0.5 * gam / beta)
        vs = vx * vx + vy * vy
        H = a * a / (gam - 1) + 0.5 * vs
        v1 = vx * uy - vy * ux
        if self.flux == ROE:
            lam = [np.abs(vn - a), np.abs(vn), np.abs(vn), np.abs(vn + a)]
        else:
            lam = [np.abs(vn) + a] * 4

        def proj(z):
            b = z[:, 0] + vx * z[:, 1] + vy * z[:, 2]
            u = a * (ux * z[:, 1] + uy * z[:, 2] + vn * z[:, 3])
            return [b + H * z[:, 3] - u, b + 0.5 * vs * z[:, 3],
                    uy * z[:, 1] - ux * z[:, 2] + v1 * z[:, 3], b + H * z[:, 3] + u]

        dz = proj(Vr - Vl)
        if d is not None:
            gl, gr = proj(d[0]), proj(d[1])
            for i in range(4):
                if self.rec == "second":
                    dz[i] = dz[i] - 0.5 * (gl[i] + gr[i])
                else:
                    j = dz[i]
                    for q in (gl[i], gr[i]):
                        b = 2 * q - j
                        mm = np.where(b * j > 0, np.sign(j) * np.minimum(np.abs(b), np.abs(j)), 0.0)
                        dz[i] = dz[i] - 0.5 * mm
        sc = [rho / (2 * gam), (gam - 1) * rho / gam, p, rho / (2 * gam)]
        z = [sc[i] * lam[i] * dz[i] for i in range(4)]
        s, d = z[0] + z[1] + z[3], z[3] - z[0]
        D = np.stack([s, vx * s + a * ux * d + uy * z[2], vy * s + a * uy * d - ux * z[2],
                      H * (z[0] + z[3]) + 0.5 * vs * z[1] + a * vn * d + v1 * z[2]], 1)
        return (F - 0.5 * D) * area[:, None]

    def viscous(self, s, dV, nx, ny):
        """Viscous flux (minus the stress and the conducted heat) through (nx, ny)
        from entropy variables s and their gradients."""
        gam, mu = self.gam, self.mu
        k = mu * gam / (gam - 1) / self.pr
        T0 = -1.0 / s[:, 3]
        u, v = s[:, 1] * T0, s[:, 2] * T0
        dT = dV[:, 3, :] * (T0 * T0)[:, None]
        du = dV[:, 1, :] * T0[:, None] + s[:, 1:2] * dT
        dv = dV[:, 2, :] * T0[:, None] + s[:, 2:3] * dT
        div = du[:, 0] + dv[:, 1]
        sxx, syy = mu * (2 * du[:, 0] - 2 / 3 * div), mu * (2 * dv[:, 1] - 2 / 3 * div)
        sxy = mu * (du[:, 1] + dv[:, 0])
        return -np.stack([0 * u, sxx * nx + sxy * ny, sxy * nx + syy * ny,
                          (u * sxx + v * sxy + k * dT[:, 0]) * nx
                          + (u * sxy + v * syy + k * dT[:, 1]) * ny], 1)

    def residual(self, w):
        g = self.g
        V = self.ent(w)
        need = self.rec != "first" and self.flux != KEPEC
        G = self.cell_gradients(w, V) if need or self.ns else None
        dV = None
        if need:
            acc = sum(g.add(g.c[:, j], G.reshape(-1, 8)) for j in range(3))
            dV = (g.gather(acc) / (6.0 * g.area[:, None])).reshape(-1, 4, 2)
        F = self.edge_flux(w, V, dV)
        R = g.add(g.l, F) - g.add(g.r, F)
        if g.nb:
            for i in (g.b0, g.b1):
                R += g.add(i, 0.5 * self.outer_flux(w, i))
        if self.ns:
            dC = G / (2.0 * g.carea)[:, None, None]
            q = ~g.wall if g.nb else np.ones(g.c.shape[0], bool)
            s = (V[g.c[q, 0]] + V[g.c[q, 1]] + V[g.c[q, 2]]) / 3.0
            for j in range(3):
                R -= g.add(g.c[q, j], 0.5 * self.viscous(s, dC[q], g.Nx[q, j], g.Ny[q, j]))
            if g.nb:
                R += self.wall_terms(w, dC)
        return g.gather(R)

    def outer_flux(self, w, i):
        """Flux through the outer edges from the states of their end points i."""
        g, gam = self.g, self.gam
        nx, ny = g.bnx, g.bny
        wi = w[i]
        s0, pb = wi.copy(), wi[:, 3].copy()
        for k in g.kinds:
            q = g.btype == k
            if k == "noslip":  # the wall's T and velocity, the fluid's pressure
                s0[q, :3] = g.bval[q, :3]
            elif k == "slip":
                s0[q] = self.one_state(k, wi[q], g.bval[q], nx[q], ny[q])
            elif k == "pressure":
                pb[q] = g.bval[q, 3]
        rho, p = s0[:, 3] / s0[:, 0], s0[:, 3]
        vn = s0[:, 1] * nx + s0[:, 2] * ny
        m = rho * vn
        F = np.stack([m, nx * pb + s0[:, 1] * m, ny * pb + s0[:, 2] * m,
                      (0.5 * rho * (s0[:, 1] ** 2 + s0[:, 2] ** 2) + gam * p / (gam - 1)) * vn
                      + (pb - p) * vn], 1)
        q = g.btype == "farfield"
        if q.any():
            F[q] = self.two_point(wi[q], g.bval[q], self.ent(wi[q]), self.ent(g.bval[q]), None,
                                  nx[q], ny[q])
        return F

    def wall_terms(self, w, dC):
        """Cells on outer edges, once per outer edge: the cell's flux from the
        edges' mean boundary state, and the wall flux at the edge's ends."""
        g = self.g
        sums, cnt = np.zeros((g.c.shape[0], 4)), np.bincount(g.bcell, minlength=g.c.shape[0])
        for i in (g.b0, g.b1):
            np.add.at(sums, g.bcell, self.ent(self.bstates(w, i, g.hx, g.hy)))
        s = sums[g.bcell] * (0.5 / cnt[g.bcell])[:, None]
        d = dC[g.bcell]
        R = np.zeros((g.nv, 4))
        for j in range(3):
            R -= g.add(g.c[g.bcell, j], 0.5 * self.viscous(s, d, g.Nx[g.bcell, j], g.Ny[g.bcell, j]))
        F = self.viscous(s, d, g.bnx, g.bny)
        slip = g.btype == "slip"  # adiabatic: no heat through it
        if slip.any():
            k = self.mu * self.gam / (self.gam - 1) / self.pr
            T0 = -1.0 / s[:, 3]
            F[:, 3] += np.where(slip, k * T0 * T0 * (d[:, 3, 0] * g.bnx + d[:, 3, 1] * g.bny), 0.0)
        for i in (g.b0, g.b1):
            R += g.add(i, 0.5 * F)
        return R

    def time_step(self, w):
        g = self.g
        c = np.sqrt(self.gam * w[:, 0])
        lam = np.zeros(g.nv)
        for i in (g.l, g.r):
            lam += np.bincount(i, np.abs(w[i, 1] * g.nx + w[i, 2] * g.ny) + c[i] * g.ar, g.nv)
        if g.nb:
            a = np.sqrt(g.bnx ** 2 + g.bny ** 2)
            for i in (g.b0, g.b1):
                lam += np.bincount(i, 0.5 * (np.abs(w[i, 1] * g.bnx + w[i, 2] * g.bny) + c[i] * a), g.nv)
        if self.ns:
            dl = np.sqrt(g.dx ** 2 + g.dy ** 2)
            for i in (g.l, g.r):
                lam += np.bincount(i, self.mu * g.ar / dl * w[i, 0] / w[i, 3], g.nv)
        return (self.cfl * g.area / g.gather(lam)).min()

    def step(self, w, t):
        """One step from (w, t): the new state, dt and the residual norm."""
        g = self.g
        dt, a = self.time_step(w), g.area[:, None]
        if self.t_end is not None and t + dt > self.t_end:
            dt = self.t_end - t
        U0 = self.con(w)
        if self.scheme == "rk4":
            Rs = []
            for c in (0.0, 0.5, 0.5, 1.0):
                wk = self.prim(U0 - dt * c / a * Rs[-1]) if Rs else w
                Rs.append(self.residual(wk))
            R = Rs[-1]
            U = U0 - dt / a / 6.0 * (Rs[0] + 2 * Rs[1] + 2 * Rs[2] + Rs[3])
        else:
            U, wk = U0, w
            for al, be in (((0, 1), (0.75, 0.25), (1 / 3, 2 / 3)) if self.scheme == "ssprk3"
                           else ((0, 1), (0.5, 0.5))):
                R = self.residual(wk)
                U = al * U0 + be * (U - dt / a * R)
                wk = self.prim(U)
        n = np.sqrt((g.weight[:, None] * (R / a) ** 2).sum(0)) / g.nv
        return self.prim(U), dt, np.sqrt((n * n).sum())

    def integrals(self, w):
        rho = w[:, 3] / w[:, 0]
        s = np.log(w[:, 3]) - self.gam * np.log(rho)
        da = self.g.area * self.g.weight
        return ((0.5 * rho * (w[:, 1] ** 2 + w[:, 2] ** 2) * da).sum(),
                (-rho * s / (self.gam - 1) * da).sum())

    def probe(self, w, px, py):
        """Density at the points, linear in the triangle that holds each."""
        g = self.g
        rho = w[:, 3] / w[:, 0]
        out = np.empty(px.size)
        for k in range(px.size):
            l = []
            for j in range(3):
                a, b = (j + 1) % 3, (j + 2) % 3
                l.append(((g.X[:, a] - px[k]) * (g.Y[:, b] - py[k])
                          - (g.X[:, b] - px[k]) * (g.Y[:, a] - py[k])) / (2 * g.carea))
            l = np.stack(l, 1)
            c = int(l.min(1).argmax())
            out[k] = (l[c] * rho[g.c[c]]).sum()
        return out


EXACT_VERTEX_STAGES = 5.0e6  # about 20 seconds of numpy


def _exact_batch(problem, mesh, inputs, flux, rec, name, t_end):
    gam = np.broadcast_to(problem.gamma(inputs), (len(next(iter(inputs.values()))),))
    Q, fields = [], []
    for k in range(gam.size):
        one = {q: float(v[k]) for q, v in inputs.items()}
        sc = _Scheme(mesh, name, flux, rec, "ssprk3", float(gam[k]), t_end)
        w, t = problem.state(mesh, one), 0.0
        while t < t_end:
            w, dt, _ = sc.step(w, t)
            t = t_end if t + dt >= t_end * (1 - 1e-15) else t + dt
        ke, ent = sc.integrals(w)
        Q.append(np.concatenate([sc.probe(w, *problem.probes), [ke, ent]]))
        fields.append(np.concatenate([w, (w[:, 3] / w[:, 0])[:, None]], 1))
    f = np.stack(fields)
    return np.stack(Q), f.mean(0), ((f - f.mean(0)) ** 2).sum(0), (f * f).sum(0)


def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("run", "watch"):
        cost = case["n"] ** 2 * case["steps"] * STAGES[case["scheme"]]
        if cost > EXACT_VERTEX_STAGES:
            return None
        m = _mesh(case["problem"], case["n"], seed)
        sc = _Scheme(m, case["problem"], case["flux"], case["rec"], case["scheme"])
        w, t, res0 = _state(case["problem"], m, rng), 0.0, None
        log, bounds = [], []
        for _ in range(case["steps"]):
            w, dt, res = sc.step(w, t)
            t += dt
            res0 = res if res0 is None else res0
            log.append((dt, res / res0, *sc.integrals(w)))
            lo, hi = w.min(0), w.max(0)
            bounds.append([lo[0], hi[0], lo[3], hi[3], lo[1], hi[1], lo[2], hi[2], 0.0, 0.0])
        if kind == "run":
            return {"steps": None, "state": w}
        return {"log": np.array(log), "bounds": np.array(bounds), "state": w}
    if kind == "batch":
        p = _problem(case)
        n, vortex = case["n"], case["problem"] == "vortex"
        steps = _steps_to(n, case["t_end"], case["problem"])
        if n * n * steps * 3 * case["samples"] > EXACT_VERTEX_STAGES:
            return None
        Q, mean, m2, s2 = _exact_batch(p, _mesh(case["problem"], n, seed),
                                       _inputs(p, case["samples"], seed), ROE if vortex else RUSANOV,
                                       case["rec"], case["problem"], case["t_end"])
        return {"qoi": Q, "mean": mean, "m2": m2, "s2": s2}
    if kind == "levels":
        p = _problem(case)
        if sum(n * n * _steps_to(n, case["t_end"]) * 3 * ns for n, ns in _levels(case)) > EXACT_VERTEX_STAGES:
            return None
        got = [_exact_batch(p, _mesh("vortex", n, seed + k), _inputs(p, ns, seed + k), ROE, "minmod",
                            "vortex", case["t_end"]) for k, (n, ns) in enumerate(_levels(case))]
        return {"qoi": [q[0] for q in got], "mean": [q[1] for q in got]}
    return _exact_net(case, seed)


def _unpack(case, p):
    w, o, out = _widths(case), 0, []
    for a, b in zip(w[:-1], w[1:]):
        out.append((p[o:o + a * b].reshape(b, a), p[o + a * b:o + a * b + b]))
        o += a * b + b
    return out


def _gelu(z):
    return 0.5 * z * (1 + torch.erf(z * 0.7071067811865476))


def _exact_net(case, seed):
    u, q, p0 = _net_inputs(case, seed)
    x = torch.from_numpy((u - u.mean(0)) / (u.std(0) + 1e-12))
    t = torch.from_numpy((q - q.mean(0)) / (q.std(0) + 1e-30))
    p = torch.from_numpy(p0.astype(np.float64)).requires_grad_(case["kind"] == "fit")

    def net(x):
        layers = _unpack(case, p)
        for k, (W, b) in enumerate(layers):
            x = x @ W.T + b
            if k + 1 < len(layers):
                x = _gelu(x)
        return x

    if case["kind"] == "predict":
        return net(x).numpy() * (q.std(0) + 1e-30) + q.mean(0)
    # minibatch Adam over the documented shuffle (a splitmix64 stream, last index first)
    mask = (1 << 64) - 1
    z = 0x5851f42d4c957f2d

    def nxt():
        nonlocal z
        z = (z + 0x9e3779b97f4a7c15) & mask
        h = ((z ^ (z >> 30)) * 0xbf58476d1ce4e5b9) & mask
        h = ((h ^ (h >> 27)) * 0x94d049bb133111eb) & mask
        return h ^ (h >> 31)

    n = case["rows"]
    perm = list(range(n))
    m, v, k, losses = torch.zeros_like(p), torch.zeros_like(p), 0, []
    for _ in range(case["epochs"]):
        for i in range(n - 1, 0, -1):
            j = nxt() % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        total = 0.0
        for b in range(0, n, case["batch"]):
            idx = torch.tensor(perm[b:b + case["batch"]])
            d = net(x[idx]) - t[idx]
            loss = (d * d).mean()
            g, = torch.autograd.grad(loss, p)
            total += float((d * d).sum())
            k += 1
            with torch.no_grad():
                m.mul_(0.9).add_(g, alpha=0.1)
                v.mul_(0.999).addcmul_(g, g, value=0.001)
                p -= 2e-3 * (m / (1 - 0.9 ** k)) / ((v / (1 - 0.999 ** k)).sqrt() + 1e-8)
        losses.append(total / (n * case["n_out"]))
    return {"loss": np.array(losses), "params": p.detach().numpy()}
