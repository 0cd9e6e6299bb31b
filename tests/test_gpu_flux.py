"""GPU: 3D divergence form marched along z against the tile kernels of the same system."""
import ctypes

import numpy as np
import pytest

import molgpu
from test_flux import SYSTEMS
from molgpu import systems
from molgpu.problem import ODEProblem

pytestmark = pytest.mark.gpu


def _dev(x, dtype):
    import torch
    return torch.tensor(np.asarray(x), dtype=torch.float64, device="cuda").to(dtype)


def _problem(sys_disc, flux, monkeypatch, tile=None):
    monkeypatch.setenv("MOL_FLUX", str(flux))
    if tile:
        monkeypatch.setenv("MOL_FLUX_TILE", tile)
        monkeypatch.setenv("MOL_FLUX_VJP_TILE", tile)
    prob = molgpu.discretize(*sys_disc) if isinstance(sys_disc, tuple) else ODEProblem(sys_disc)
    rng = np.random.default_rng(5)
    for a in prob.lowered.aux:
        prob.set_grid_field(a, rng.uniform(0.5, 1.5, prob.lowered.n))
    prob.handle
    return prob


def _both(prob, t):
    import torch
    td = prob.torch_dtype()
    N = prob.lowered.n_unknowns
    rng = np.random.default_rng(7)
    u, lam = _dev(rng.uniform(-0.8, 0.8, N), td), _dev(rng.standard_normal(N), td)
    out = torch.empty_like(u)
    prob.f(out, u, None, t)
    g = torch.zeros(max(1, len(prob.lowered.aux)) * int(np.prod(prob.lowered.n)), dtype=torch.float64, device="cuda")
    vjp = prob.vjp(u, lam, t, g_aux=g if prob.lowered.aux else None)
    torch.cuda.synchronize()
    return [v.double().cpu().numpy() for v in (out, vjp, g)]


# tiles and chunks that leave remainders, the sizes that the rule takes, FP32 and FP64
@pytest.mark.parametrize("n,tile", [(12, "8,8,3"), (19, "16,16,5"), (35, "32,8,4"), (51, "32,16,64"), (54, None), (75, None)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_march_equals_tiles(n, tile, dtype, monkeypatch):
    print("  flux n=%d %s tile=%s" % (n, dtype, tile), flush=True)
    ref = _both(_problem(systems.nonlindiff3d(n, dtype=dtype), 0, monkeypatch), 0.0)
    got = _both(_problem(systems.nonlindiff3d(n, dtype=dtype), 1, monkeypatch, tile), 0.0)
    # some fifty roundings of terms of the size of the largest result
    tol = 1e-13 if dtype == "f64" else 1e-5
    for a, b in zip(got, ref):
        assert np.max(np.abs(a - b)) <= tol * np.max(np.abs(b))


@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_march_of_other_systems(name, monkeypatch):
    print("  flux %s" % name, flush=True)
    ref = _both(_problem(SYSTEMS[name](), 0, monkeypatch), 0.4)
    got = _both(_problem(SYSTEMS[name](), 1, monkeypatch), 0.4)
    for a, b in zip(got, ref):
        assert np.max(np.abs(a - b)) <= 1e-13 * (np.max(np.abs(b)) + 1e-300)


@pytest.mark.parametrize("steps,every", [(1, 0), (4, 2), (5, 2)])
def test_adjoint_and_steps(steps, every, monkeypatch):
    """Whole steps (both update epilogues and the graph), the adjoint over an odd and an even number
    of steps, twice in a row."""
    import torch
    n, dt = 23, 1e-5
    res = []
    for flux in (0, 1):
        prob = _problem(systems.nonlindiff3d(n), flux, monkeypatch)
        N = prob.lowered.n_unknowns
        rng = np.random.default_rng(2)
        u0, lam0 = rng.uniform(-0.5, 0.5, N), rng.standard_normal(N)
        r = []
        for kw in ({}, {"graph": True}, {"kahan": True}):
            u = _dev(u0, torch.float64)
            prob.integrate(u, 0.0, dt, 2 * steps + 1, molgpu.RK4, **kw)
            r.append(u)
        for rep in range(2):
            print("  flux adjoint steps=%d every=%d flux=%d rep=%d" % (steps, every, flux, rep), flush=True)
            u, lam = _dev(u0, torch.float64), _dev(lam0, torch.float64)
            g = torch.zeros(2 * n ** 3, dtype=torch.float64, device="cuda")
            prob.forward_checkpointed(u, 0.0, dt, steps, every)
            prob.adjoint(lam, g_aux=g)
            r += [u, lam, g]
        torch.cuda.synchronize()
        res.append([v.cpu().numpy() for v in r])
    for a, b in zip(*res):
        assert np.max(np.abs(b - a)) <= 1e-12 * np.max(np.abs(a))


def test_result_over_its_own_seed(monkeypatch):
    """lam_dot may be lam itself (or the state), as with the tile kernels."""
    import torch
    prob = _problem(systems.nonlindiff3d(30), 1, monkeypatch)
    N = prob.lowered.n_unknowns
    rng = np.random.default_rng(3)
    u, lam = _dev(rng.uniform(-1, 1, N), torch.float64), _dev(rng.standard_normal(N), torch.float64)
    ref = prob.vjp(u, lam)
    h = prob.handle
    for over in (lam, u):
        a, b = u.clone(), lam.clone()
        out = b if over is lam else a
        rc = h.lib.mol_vjp(h.h, a.data_ptr(), None, 0.0, b.data_ptr(), out.data_ptr(), None,
                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        torch.cuda.synchronize()
        assert torch.equal(out, ref)


@pytest.mark.parametrize("n,steps,every", [(12, 5, 2), (12, 4, 9), (19, 6, 3)])
def test_second_adjoint_of_a_run(n, steps, every, monkeypatch):
    """The first sweep of a run uses the stage states of its last segment, later ones recompute
    them: same bits, and those of a run that kept every state."""
    import torch
    prob = _problem(systems.nonlindiff3d(n), 1, monkeypatch)
    N = prob.lowered.n_unknowns
    rng = np.random.default_rng(4)
    u0, lam0 = _dev(rng.uniform(-1, 1, N), torch.float64), _dev(rng.standard_normal(N), torch.float64)
    res = []
    for ev in (0, every):
        u = u0.clone()
        print("  flux second adjoint n=%d every=%d" % (n, ev), flush=True)
        prob.forward_checkpointed(u, 0.0, 1e-5, steps, ev)
        for rep in range(1 if ev == 0 else 3):
            lam = lam0.clone()
            g = torch.zeros(2 * n ** 3, dtype=torch.float64, device="cuda")
            prob.adjoint(lam, g_aux=g)
            res.append((u, lam, g))
    torch.cuda.synchronize()
    for r in res[1:]:
        for a, b in zip(r, res[0]):
            assert torch.equal(a, b)


@pytest.mark.parametrize("n", [42, 43, 49, 50])
def test_sizes_at_the_lines_of_the_rule(n, monkeypatch):
    """Tiles in both directions, march in the reverse direction only, march in both."""
    import torch
    steps, dt = 3, 1e-6
    res = []
    for flux in ("0", None):
        if flux is None:
            monkeypatch.delenv("MOL_FLUX", raising=False)
        else:
            monkeypatch.setenv("MOL_FLUX", flux)
        prob = molgpu.discretize(*systems.nonlindiff3d(n))
        rng = np.random.default_rng(n)
        for a in prob.lowered.aux:
            prob.set_grid_field(a, rng.uniform(0.5, 1.5, prob.lowered.n))
        N = prob.lowered.n_unknowns
        u, lam = _dev(rng.uniform(-0.5, 0.5, N), torch.float64), _dev(rng.standard_normal(N), torch.float64)
        g = torch.zeros(2 * n ** 3, dtype=torch.float64, device="cuda")
        print("  flux rule n=%d flux=%s" % (n, flux), flush=True)
        prob.forward_checkpointed(u, 0.0, dt, steps, 2)
        prob.adjoint(lam, g_aux=g)
        torch.cuda.synchronize()
        res.append([v.cpu().numpy() for v in (u, lam, g)])
    for a, b in zip(*res):
        assert np.max(np.abs(b - a)) <= 1e-12 * np.max(np.abs(a))
