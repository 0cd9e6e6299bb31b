"""The calls that programs built on this framework spend their time in.

Eight kinds of work, each through the package's public entry points, from the smallest systems
(where the latency of a call counts) to grids that fill the card:

  heat           ``solve`` of the 1D heat equation with saved states: thousands of small steps
  bruss_rhs      one ``f(du, u, p, t)`` of the 2D Brusselator, as an integrator of the caller's
                 own calls it once per stage
  bruss          fixed-step RK4 of the 2D Brusselator (``ODEProblem.integrate``)
  burgers        fixed-step SSPRK33 of the WENO5 Burgers system, FP64, or FP32 with the compensated
                 update
  burgers_rhs    one right-hand side of the WENO5 Burgers system, on uniform or stretched nodes
  nonlin         fixed-step RK4 of 3D nonlinear diffusion with grid-valued coefficients
  nonlin_grad    ``rk4_solve`` of that system and the gradients of a misfit with respect to the
                 initial state and the two coefficient fields (forward and backward)
  batch          fixed-step RK4 of many uneven diffusion-reaction instances, FP32 with the
                 compensated update (``BatchProblem.integrate``)

A pass of an integration restarts from the case's initial state, so passes repeat the same work.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "methodoflines.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import molgpu  # noqa: E402
from molgpu import systems  # noqa: E402
from molgpu.autograd import rk4_solve  # noqa: E402
from molgpu.batch import BatchProblem  # noqa: E402

DEVICE = "cuda"


def listed():
    return [
        # the smallest solve: 101 nodes, 10000 RK4 steps of 1e-5 to t = 0.1, ten saved states
        {"name": "heat 101 solve", "kind": "heat", "n": 101, "steps": 10000, "saves": 10, "dt": 1e-5,
         "left": "dirichlet", "right": "dirichlet"},
        # the smallest call: one right-hand side of a coarse grid
        {"name": "brusselator 64 rhs", "kind": "bruss_rhs", "n": 64},
        # the ordinary 2D solve, 20 RK4 steps of 512 x 512 x 2 unknowns
        {"name": "brusselator 512 rk4", "kind": "bruss", "n": 512, "steps": 20},
        # a grid beyond one tile per compute unit, odd size
        {"name": "brusselator 1501 rk4", "kind": "bruss", "n": 1501, "steps": 4},
        # WENO5 in the stage loop, FP64
        {"name": "burgers 1024 ssprk3", "kind": "burgers", "n": 1024, "steps": 4, "dtype": "f64"},
        # the same in the FP32 mode with compensated updates, odd size
        {"name": "burgers 1447 f32 ssprk3", "kind": "burgers", "n": 1447, "steps": 4, "dtype": "f32"},
        # WENO5 far beyond the caches
        {"name": "burgers 4096 rhs", "kind": "burgers_rhs", "n": 4096, "stretched": False},
        # WENO5 on stretched node arrays along both axes
        {"name": "burgers 1024 stretched rhs", "kind": "burgers_rhs", "n": 1024, "stretched": True},
        # 3D forward run
        {"name": "nonlinear 128 rk4", "kind": "nonlin", "n": 128, "steps": 4, "dtype": "f64"},
        # 3D forward and backward, every stage state kept
        {"name": "nonlinear 128 gradient", "kind": "nonlin_grad", "n": 128, "steps": 5, "every": 0, "dtype": "f64"},
        # the same on an odd grid in FP32 with checkpoints and recomputed segments
        {"name": "nonlinear 75 f32 gradient", "kind": "nonlin_grad", "n": 75, "steps": 24, "every": 8, "dtype": "f32"},
        # many instances of 32 .. 256 nodes per side in one state vector
        {"name": "batch 512 f32 rk4", "kind": "batch", "count": 512, "steps": 4, "sizes": 2024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["heat", "bruss_rhs", "bruss", "burgers", "burgers_rhs", "nonlin", "nonlin_grad", "batch"])
    if kind == "heat":
        n = _log(rng, 24, 700)
        steps = _log(rng, 200, 6000)
        return {"kind": kind, "n": n, "steps": steps, "saves": rng.choice([1, 2, 5, 10]),
                "dt": 0.3 / (n - 1) ** 2, "left": rng.choice(["dirichlet", "neumann"]),
                "right": rng.choice(["dirichlet", "neumann"])}
    if kind == "bruss_rhs":
        return {"kind": kind, "n": _not5(_log(rng, 24, 1600))}
    if kind == "bruss":
        n = _not5(_log(rng, 48, 1600))
        return {"kind": kind, "n": n, "steps": max(1, min(25, int(6e6 / n ** 2)) - rng.randrange(2))}
    if kind == "burgers":
        n = _log(rng, 96, 2000)
        return {"kind": kind, "n": n, "steps": max(1, min(12, int(4e6 / n ** 2))), "dtype": rng.choice(["f64", "f32"])}
    if kind == "burgers_rhs":
        stretched = rng.random() < 0.5
        return {"kind": kind, "n": _log(rng, 128, 1024 if stretched else 3500), "stretched": stretched}
    if kind == "nonlin":
        n = rng.randrange(24, 129)
        return {"kind": kind, "n": n, "steps": rng.randrange(1, 5), "dtype": rng.choice(["f64", "f32"])}
    if kind == "nonlin_grad":
        n = rng.randrange(20, 100)
        return {"kind": kind, "n": n, "steps": rng.randrange(2, 9), "every": rng.choice([0, 3, 20]),
                "dtype": rng.choice(["f64", "f32"])}
    return {"kind": kind, "count": _log(rng, 4, 300), "steps": rng.randrange(1, 6), "sizes": rng.randrange(1, 10 ** 6)}


def _not5(n):
    # the forcing of the Brusselator switches on a disc whose rim holds grid nodes exactly when
    # n is a multiple of 5; there the last bit of a coordinate decides
    return n + 1 if n % 5 == 0 else n


# ------------------------------------------------------------------ inputs (made from the seed)
def _gen(seed, device):
    return torch.Generator(device=device).manual_seed(int(seed))


def _rand(g, shape, device):
    return torch.rand(shape, generator=g, dtype=torch.float64, device=device)


def _host(seed, *shape):
    return np.random.default_rng(int(seed)).random(shape)


def _heat_u0(case, seed):
    a = _host(seed, 6)
    x = np.arange(case["n"]) / (case["n"] - 1.0)
    u = sum((a[k] - 0.3) / (k + 1) * np.sin((k + 1) * math.pi * x) for k in range(6))
    return u[1:-1]


def _bruss_state(case, seed, device):
    n = case["n"]
    ph = _host(seed, 8)
    c = torch.arange(1, n + 1, dtype=torch.float64, device=device) / n
    y, x = c[:, None], c[None, :]
    ripple = lambda k: 1 + 0.1 * torch.cos(2 * math.pi * (x + ph[k])) * torch.cos(4 * math.pi * (y + ph[k + 1]))
    u = 0.4 + 22 * (y * (1 - y)).abs() ** 1.5 * ripple(0)
    v = 0.4 + 27 * (x * (1 - x)).abs() ** 1.5 * ripple(2)
    return torch.stack([u, v])


def _bruss_dt(case):
    return 0.1 / (10.0 * case["n"] ** 2)


BRUSS_T0 = 1.2    # the forcing is on


def _axis_nodes(case, axis):
    if not case.get("stretched"):
        return None
    n = case["n"] + 1
    h = 1.0 + 0.3 * (2 * _host(17 + axis, n - 1) - 1)
    x = np.concatenate([[0.0], np.cumsum(h)])
    x = x / x[-1]
    x[-1] = 1.0
    return x


def _burgers_state(case, seed, device):
    n = case["n"]
    p = _host(seed, 8, 4)
    xs = []
    for a in range(2):
        nodes = _axis_nodes(case, a)
        xs.append(torch.arange(1, n + 1, dtype=torch.float64, device=device) / n if nodes is None
                  else torch.tensor(nodes[1:], device=device))
    x, y = xs[0][None, :], xs[1][:, None]
    u = torch.full((n, n), 0.5, dtype=torch.float64, device=device)
    for cx, cy, w, a in p:
        dx, dy = (x - cx).abs(), (y - cy).abs()
        dx, dy = torch.minimum(dx, 1 - dx), torch.minimum(dy, 1 - dy)
        s = -1.0 / (2 * (0.02 + 0.06 * w) ** 2)
        u += (0.1 + 0.4 * a) * torch.exp(s * dx * dx) * torch.exp(s * dy * dy)
    return u


def _burgers_dt(case):
    return 0.1 / case["n"]


def _nonlin_inputs(case, seed, device):
    """u0, target over the unknowns and d0, s over the grid (z, y, x), FP32 values in FP32 cases."""
    n = case["n"]
    c = torch.arange(n, dtype=torch.float64, device=device) / (n - 1)

    def field(k):
        p = _host(int(seed) * 8 + k, 8, 5)
        out = torch.zeros((n, n, n), dtype=torch.float64, device=device)
        for cx, cy, cz, w, a in p:
            s = -1.0 / (2 * (0.08 + 0.15 * w) ** 2)
            ex, ey, ez = (torch.exp(s * (c - q) ** 2) for q in (cx, cy, cz))
            out += (2 * a - 1) * ez[:, None, None] * ey[None, :, None] * ex[None, None, :]
        return out

    inner = slice(1, n - 1)
    u0, tgt = (f[inner, inner, inner].contiguous() for f in (0.3 * field(0), 0.2 * field(1)))
    got = [u0, tgt, 0.5 + 0.5 * field(2).abs(), field(3)]
    if case["dtype"] == "f32":
        got = [f.float().double() for f in got]
    return got


def _nonlin_dt(case):
    return 0.02 / (case["n"] - 1) ** 2


def _batch_instances(case):
    r = np.random.default_rng(case["sizes"])
    got = []
    for _ in range(case["count"]):
        got.append((int(r.integers(32, 257)), float(r.uniform(0.01, 0.1)), float(r.uniform(0.5, 5.0)),
                    tuple(int(b) for b in r.integers(0, 2, 4))))
    return got


def _batch_dt(case):
    return min(0.5 * 2.78 / ((n - 1) ** 2 * 8 * D) for n, D, _, _ in _batch_instances(case))


def _batch_state(case, seed, device):
    total = sum((n - 2) ** 2 for n, _, _, _ in _batch_instances(case))
    return 0.1 + 0.8 * _rand(_gen(seed, device), (total,), device)


# ------------------------------------------------------------------ the framework's side
def _burgers_system(case, dtype):
    t, x, y = molgpu.parameters("t x y")
    u = molgpu.variables("u")
    Dt, Dx, Dy = molgpu.Differential(t), molgpu.Differential(x), molgpu.Differential(y)
    U = u(t, x, y)
    eq = molgpu.Eq(Dt(U), -U * Dx(U) - U * Dy(U))
    bcs = [molgpu.Eq(u(0, x, y), 0.5), molgpu.Eq(u(t, 0, y), u(t, 1, y)), molgpu.Eq(u(t, x, 0), u(t, x, 1))]
    sys_ = molgpu.PDESystem([eq], bcs, [molgpu.Interval(v, 0.0, 1.0) for v in (t, x, y)], [t, x, y], [U])
    nodes = [_axis_nodes(case, a) for a in range(2)]
    grid = {v: case["n"] + 1 if g is None else g for v, g in zip((x, y), nodes)}
    return molgpu.discretize(sys_, molgpu.MOLFiniteDifference(grid, t, advection_scheme=molgpu.WENOScheme(1e-6),
                                                              dtype=dtype))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "heat":
        bc = {"dirichlet": (1.0, 0.0, 0.0), "neumann": (0.0, 1.0, 0.0)}
        prob = molgpu.discretize(*systems.heat1d(case["n"], 1.0, bc[case["left"]], bc[case["right"]]))
        prob.u0 = _heat_u0(case, seed)
        prob.handle
        return {"case": case, "prob": prob}
    if kind in ("bruss_rhs", "bruss"):
        prob = molgpu.discretize(*systems.brusselator2d(case["n"] + 1))
        u0 = _bruss_state(case, seed, DEVICE).reshape(-1)
    elif kind in ("burgers", "burgers_rhs"):
        prob = _burgers_system(case, case.get("dtype", "f64"))
        u0 = _burgers_state(case, seed, DEVICE).reshape(-1).to(prob.torch_dtype())
    elif kind in ("nonlin", "nonlin_grad"):
        prob = molgpu.discretize(*systems.nonlindiff3d(case["n"], dtype=case["dtype"]))
        u0, tgt, d0, s = (f.reshape(-1).to(prob.torch_dtype()) for f in _nonlin_inputs(case, seed, DEVICE))
        prob.set_grid_field("d0", d0)
        prob.set_grid_field("s", s)
        if kind == "nonlin_grad":
            prob.handle
            leaves = [f.clone().requires_grad_() for f in (u0, d0, s)]
            return {"case": case, "prob": prob, "leaves": leaves, "tgt": tgt}
    else:
        lows = [molgpu.lower(*systems.diffreact2d(n, D, k, bc, dtype="f32"))
                for n, D, k, bc in _batch_instances(case)]
        prob = BatchProblem(lows, tile=(256, 16, 1))    # the tile that the tuner finds for such batches
        u0 = _batch_state(case, seed, DEVICE).float()
        return {"case": case, "prob": prob, "u0": u0, "u": u0.clone(), "dt": _batch_dt(case)}
    prob.handle
    return {"case": case, "prob": prob, "u0": u0, "u": torch.empty_like(u0)}


def run(state):
    case, prob = state["case"], state["prob"]
    kind = case["kind"]
    if kind == "heat":
        every = case["steps"] // case["saves"]
        sol = molgpu.solve(prob, molgpu.RK4, dt=case["dt"], saveat=every * case["dt"],
                           tspan=(0.0, case["steps"] * case["dt"]))
        return sol["u"]
    if kind in ("bruss_rhs", "burgers_rhs"):
        prob.f(state["u"], state["u0"], None, BRUSS_T0)
        return state["u"]
    if kind == "nonlin_grad":
        u0, d0, s = state["leaves"]
        u = rk4_solve(prob, u0, 0.0, _nonlin_dt(case), case["steps"], ckpt_every=case["every"],
                      grid_fields={"d0": d0, "s": s})
        misfit = 0.5 * ((u - state["tgt"]) ** 2).sum()
        return [u.detach(), *torch.autograd.grad(misfit, [u0, d0, s])]
    u = state["u"]
    u.copy_(state["u0"])
    if kind == "bruss":
        prob.integrate(u, BRUSS_T0, _bruss_dt(case), case["steps"])
    elif kind == "burgers":
        prob.integrate(u, 0.0, _burgers_dt(case), case["steps"], molgpu.SSPRK33, kahan=case["dtype"] == "f32")
    elif kind == "nonlin":
        prob.integrate(u, 0.0, _nonlin_dt(case), case["steps"])
    else:
        prob.integrate(u, 0.0, state["dt"], case["steps"], kahan=True)
    return u


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind = case["kind"]
    es = 4 if case.get("dtype") == "f32" or kind == "batch" else 8
    n, steps = case.get("n", 0), case.get("steps", 1)
    if kind == "heat":     # 5 operations per node and stage, 3 of the update
        return {"bytes": 8.0 * (n + n * (case["saves"] + 1)), "flops": 8.0 * 4 * steps * (n - 2)}
    if kind == "bruss_rhs":
        return {"bytes": 32.0 * n * n, "flops": 30.0 * n * n}
    if kind == "bruss":
        return {"bytes": 32.0 * n * n, "flops": 38.0 * 4 * steps * n * n}
    if kind == "burgers":  # two WENO5 derivatives of about 60 operations per node and stage
        return {"bytes": 2.0 * es * n * n, "flops": 127.0 * 3 * steps * n * n}
    if kind == "burgers_rhs":
        return {"bytes": 16.0 * n * n, "flops": (230.0 if case["stretched"] else 123.0) * n * n}
    if kind == "nonlin":   # 3 half-point fluxes of about 20 operations per node and stage
        return {"bytes": 4.0 * es * n ** 3, "flops": 70.0 * 4 * steps * n ** 3}
    if kind == "nonlin_grad":
        return {"bytes": 8.0 * es * n ** 3, "flops": 240.0 * 4 * steps * n ** 3}
    pts = sum((m - 2) ** 2 for m, _, _, _ in _batch_instances(case))
    return {"bytes": 8.0 * pts, "flops": 18.0 * 4 * steps * pts}


# ------------------------------------------------------------------ the same in plain FP64
def _rk4(f, u, t, dt, steps):
    for _ in range(steps):
        k1 = f(u, t)
        k2 = f(u + dt / 2 * k1, t + dt / 2)
        k3 = f(u + dt / 2 * k2, t + dt / 2)
        k4 = f(u + dt * k3, t + dt)
        u = u + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
        t = t + dt
    return u


def _heat_exact(case, seed):
    n, dt = case["n"], case["dt"]
    h2 = (n - 1.0) ** 2
    w = np.zeros(n)
    w[1:-1] = _heat_u0(case, seed)

    def ends(v):    # u = 0, or the second-order one-sided u_x = 0
        v[0] = 0.0 if case["left"] == "dirichlet" else (4 * v[1] - v[2]) / 3
        v[-1] = 0.0 if case["right"] == "dirichlet" else (4 * v[-2] - v[-3]) / 3
        return v

    def f(u, _t):
        v = np.zeros(n)
        v[1:-1] = u
        ends(v)
        return (v[:-2] - 2 * v[1:-1] + v[2:]) * h2

    every = case["steps"] // case["saves"]
    marks = list(range(every, case["steps"] + 1, every))
    if marks[-1] != case["steps"]:
        marks.append(case["steps"])
    out, done = [ends(w.copy())], 0
    u = w[1:-1].copy()
    for m in marks:
        u = _rk4(f, u, 0.0, dt, m - done)
        done = m
        v = np.zeros(n)
        v[1:-1] = u
        out.append(ends(v))
    return np.stack(out)


def _bruss_f(n, device):
    c = torch.arange(1, n + 1, dtype=torch.float64, device=device) / n
    y, x = c[:, None], c[None, :]
    disc = ((x - 0.3) ** 2 + (y - 0.6) ** 2 <= 0.1 ** 2).double()

    def lap(w):
        return (w.roll(1, 0) + w.roll(-1, 0) + w.roll(1, 1) + w.roll(-1, 1) - 4 * w) * float(n * n)

    def f(s, t):
        u, v = s[0], s[1]
        fo = disc * (5.0 if t >= 1.1 else 0.0)
        return torch.stack([1.0 + v * u * u - 4.4 * u + 10.0 * lap(u) + fo, 3.4 * u - v * u * u + 10.0 * lap(v)])

    return f


def _weno_uniform(u, axis, dx, eps):
    """Derivative by Jiang-Shu WENO5 point reconstructions at the two half points of a node."""
    a, b, c, d, e = (u.roll(k, axis) for k in (2, 1, 0, -1, -2))
    b1 = 13 * (c - 2 * d + e) ** 2 / 12 + (3 * c - 4 * d + e) ** 2 / 4
    b2 = 13 * (b - 2 * c + d) ** 2 / 12 + (b - d) ** 2 / 4
    b3 = 13 * (a - 2 * b + c) ** 2 / 12 + (a - 4 * b + 3 * c) ** 2 / 4
    r1, r2, r3 = (1 / (eps + q) ** 2 for q in (b1, b2, b3))
    m1, m2, m3 = 0.1 * r1, 0.6 * r2, 0.3 * r3
    p1, p2, p3 = 0.3 * r1, 0.6 * r2, 0.1 * r3
    hm = (m1 * (11 * c - 7 * d + 2 * e) + m2 * (2 * b + 5 * c - d) + m3 * (5 * b + 2 * c - a)) / (6 * (m1 + m2 + m3))
    hp = (p1 * (2 * c + 5 * d - e) + p2 * (5 * c + 2 * d - b) + p3 * (11 * c - 7 * b + 2 * a)) / (6 * (p1 + p2 + p3))
    return (hp - hm) / dx


def _weno_stretched(u, axis, nodes, eps):
    """Node-centred WENO5 derivative on stretched periodic nodes: three quadratics, smoothness by
    Simpson's rule over the node's cell, ideal weights of the five-point derivative, split with
    theta = 3."""
    x = np.asarray(nodes)
    n = len(x)
    period = x[-1] - x[0]
    ring = x[1:]
    m = n - 1
    at = [np.roll(ring, -k) + (period * (np.arange(m) + k >= m) - period * (np.arange(m) + k < 0))
          for k in (-2, -1, 0, 1, 2)]
    shape = (1, m) if axis == 1 else (m, 1)
    put = lambda w: torch.tensor(np.ascontiguousarray(w), device=u.device).reshape(shape)
    vals = [u.roll(k, axis) for k in (2, 1, 0, -1, -2)]
    xl, xr = (at[1] + at[2]) / 2, (at[2] + at[3]) / 2
    xm, dx = (xl + xr) / 2, xr - xl
    r, al = [], []
    for k in range(3):
        a, b, c = at[k:k + 3]
        v = vals[k:k + 3]
        la, lb, lc = 1 / ((a - b) * (a - c)), 1 / ((b - a) * (b - c)), 1 / ((c - a) * (c - b))
        d1 = lambda z: sum(put(w) * q for w, q in zip(((2 * z - b - c) * la, (2 * z - a - c) * lb, (2 * z - a - b) * lc), v))
        d2 = sum(put(2 * w) * q for w, q in zip((la, lb, lc), v))
        i1 = put(dx / 6) * (d1(xl) ** 2 + 4 * d1(xm) ** 2 + d1(xr) ** 2)
        beta = put(dx) * i1 + put(dx ** 3) * put(dx) * d2 ** 2
        r.append(d1(at[2]))
        al.append(1 / (eps + beta) ** 2)
    x1, x2, x3, x4, x5 = at
    g0 = ((x3 - x4) * (x3 - x5)) / ((x1 - x4) * (x1 - x5))
    g2 = ((x3 - x1) * (x3 - x2)) / ((x5 - x1) * (x5 - x2))
    gs = [g0, 1 - g0 - g2, g2]
    plus = [0.5 * (g + 3 * np.abs(g)) for g in gs]
    minus = [p - g for p, g in zip(plus, gs)]
    total = 0.0
    for w, sign in ((plus, 1.0), (minus, -1.0)):
        s = sum(w)
        om = [put(q / s) * a for q, a in zip(w, al)]
        total = total + sign * put(s) * sum(o * q for o, q in zip(om, r)) / sum(om)
    return total


def _burgers_f(case):
    n = case["n"]
    if case.get("stretched"):
        ax = [_axis_nodes(case, a) for a in range(2)]
        return lambda u, t: -u * (_weno_stretched(u, 1, ax[0], 1e-6) + _weno_stretched(u, 0, ax[1], 1e-6))
    return lambda u, t: -u * (_weno_uniform(u, 1, 1.0 / n, 1e-6) + _weno_uniform(u, 0, 1.0 / n, 1e-6))


def _ssprk3(f, u, dt, steps):
    for _ in range(steps):
        y = u + dt * f(u, 0.0)
        y = 0.75 * u + 0.25 * (y + dt * f(y, 0.0))
        u = u / 3 + 2.0 / 3.0 * (y + dt * f(y, 0.0))
    return u


def _half(v, axis):
    """Cubic interpolation to the half points of an axis, one-sided at its ends."""
    n = v.shape[axis]
    s = lambda a, b: v.narrow(axis, a, b - a)
    mid = (9 * (s(1, n - 2) + s(2, n - 1)) - s(0, n - 3) - s(3, n)) / 16
    lo = (5 * s(0, 1) + 15 * s(1, 2) - 5 * s(2, 3) + s(3, 4)) / 16
    hi = (5 * s(n - 1, n) + 15 * s(n - 2, n - 1) - 5 * s(n - 3, n - 2) + s(n - 4, n - 3)) / 16
    return torch.cat([lo, mid, hi], axis)


def _nonlin_f(n, d0, src):
    h = float(n - 1)

    def f(u, _t):
        out = src[1:-1, 1:-1, 1:-1]
        for a in range(3):
            m = n - 2
            s = lambda i: u.narrow(a, i, 1)
            line = torch.cat([(4 * s(0) - s(1)) / 3, u, (4 * s(m - 1) - s(m - 2)) / 3], a)
            d = d0
            for b in range(3):
                if b != a:
                    d = d.narrow(b, 1, m)
            flux = _half(d, a) * (1 + _half(line, a) ** 2) * line.diff(dim=a) * h
            out = out + flux.diff(dim=a) * h
        return out

    return f


def exact(case, seed):
    kind = case["kind"]
    device = DEVICE if torch.cuda.is_available() else "cpu"
    if kind == "heat":
        return _heat_exact(case, seed)
    if kind == "bruss_rhs":
        return _bruss_f(case["n"], device)(_bruss_state(case, seed, device), BRUSS_T0).reshape(-1)
    if kind == "bruss":
        u = _rk4(_bruss_f(case["n"], device), _bruss_state(case, seed, device), BRUSS_T0, _bruss_dt(case), case["steps"])
        return u.reshape(-1)
    if kind == "burgers":
        u0 = _burgers_state(case, seed, device)
        if case["dtype"] == "f32":
            u0 = u0.float().double()
        return _ssprk3(_burgers_f(case), u0, _burgers_dt(case), case["steps"]).reshape(-1)
    if kind == "burgers_rhs":
        return _burgers_f(case)(_burgers_state(case, seed, device), 0.0).reshape(-1)
    if kind in ("nonlin", "nonlin_grad"):
        u0, tgt, d0, s = _nonlin_inputs(case, seed, device)
        if kind == "nonlin":
            return _rk4(_nonlin_f(case["n"], d0, s), u0, 0.0, _nonlin_dt(case), case["steps"]).reshape(-1)
        leaves = [f.requires_grad_() for f in (u0, d0, s)]
        u = _rk4(_nonlin_f(case["n"], d0, s), u0, 0.0, _nonlin_dt(case), case["steps"])
        grads = torch.autograd.grad(0.5 * ((u - tgt) ** 2).sum(), leaves)
        return [f.detach().reshape(-1) for f in (u, *grads)]
    u0 = _batch_state(case, seed, device).float().double()
    dt, out, at = _batch_dt(case), [], 0
    for n, D, k, bc in _batch_instances(case):
        m = n - 2
        h2 = float((n - 1) ** 2)

        def f(u, _t):
            ghost = lambda axis, i, j, kind: torch.zeros_like(u.narrow(axis, 0, 1)) if kind == 0 else \
                (4 * u.narrow(axis, i, 1) - u.narrow(axis, j, 1)) / 3
            lx = torch.cat([ghost(1, 0, 1, bc[0]), u, ghost(1, m - 1, m - 2, bc[1])], 1).diff(n=2, dim=1)
            ly = torch.cat([ghost(0, 0, 1, bc[2]), u, ghost(0, m - 1, m - 2, bc[3])], 0).diff(n=2, dim=0)
            return D * h2 * (lx + ly) + k * u * (1 - u)

        out.append(_rk4(f, u0[at:at + m * m].reshape(m, m), 0.0, dt, case["steps"]).reshape(-1))
        at += m * m
    return torch.cat(out)
