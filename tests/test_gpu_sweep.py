"""GPU: RK4 steps of 2D systems and of batches swept along y in registers."""
import numpy as np
import pytest

import molgpu
from molgpu import systems
from molgpu.batch import BatchProblem
from molgpu.discretization import MOLFiniteDifference, UpwindScheme, lower
from molgpu.pdesys import Differential, Eq, Interval, PDESystem, parameters, variables
from test_sweep import axis_system, coupled_system

pytestmark = pytest.mark.gpu


def _run(prob, u0, t0, dt, N, **kw):
    import torch
    td = prob.torch_dtype()
    u = torch.tensor(u0, device="cuda").to(td)
    prob.integrate(u, t0, dt, N, molgpu.RK4, **kw)
    torch.cuda.synchronize()
    return u.double().cpu().numpy()


# unknowns per axis at the edges of a window: less than one, one exactly, one column more, the
# last two-window size, the first three-window size
@pytest.mark.parametrize("n,rows", [(10, 4), (57, 5), (66, 9), (67, 64), (122, 16), (123, 7)])
@pytest.mark.parametrize("case", ["periodic", (0, 1, 1, 0), (1, 0, 0, 1)])
def test_swept_steps_equal_stage_launches(case, n, rows, monkeypatch):
    monkeypatch.setenv("MOL_SWEEP", "1")
    monkeypatch.setenv("MOL_SWEEP_ROWS", str(rows))
    if case == "periodic":
        prob = molgpu.discretize(*systems.brusselator2d(n=n))
        dt, t0 = 0.01 / (n - 1) ** 2, 1.2
    else:
        prob = molgpu.discretize(*systems.diffreact2d(n, 0.1, 2.0, case))
        dt, t0 = 0.5 / (n - 1) ** 2, 0.0
    u0 = np.random.default_rng(n).uniform(0.5, 1.5, prob.lowered.n_unknowns)
    print("  sweep %s n=%d rows=%d" % (case, n, rows), flush=True)
    ref = _run(prob, u0, t0, dt, 5, fused=False)
    got = _run(prob, u0, t0, dt, 5)
    assert np.max(np.abs(got - ref)) <= 1e-13 * (1 + np.max(np.abs(ref)))


@pytest.mark.parametrize("graph", [False, True])
def test_swept_compensated_fp32_steps(graph):
    """200 FP32 steps with the compensated update stay within two roundings of the FP64 run, called
    twice (the compensation starts from zero each time); without it the error is larger."""
    n, N = 400, 200
    sy = lambda dtype: systems.diffreact2d(n, 0.05, 1.0, (0, 1, 1, 0), dtype=dtype)
    u0 = np.random.default_rng(3).uniform(0.1, 0.9, (n - 2) ** 2).astype(np.float32).astype(np.float64)
    dt = 1.0 / (n - 1) ** 2
    ref = _run(molgpu.discretize(*sy("f64")), u0, 0.0, dt, N)
    prob = molgpu.discretize(*sy("f32"))
    for call in range(2):
        print("  sweep kahan graph=%s call=%d" % (graph, call), flush=True)
        got = _run(prob, u0, 0.0, dt, N, kahan=True, graph=graph)
        stage = _run(prob, u0, 0.0, dt, N, kahan=True, graph=graph, fused=False)
        assert np.max(np.abs(got - ref)) <= 2 * np.max(np.abs(stage - ref)) + 2 ** -24
        assert np.max(np.abs(got - ref)) < np.max(np.abs(_run(prob, u0, 0.0, dt, N) - ref))


@pytest.mark.parametrize("dtype,kahan", [("f32", True), ("f32", False), ("f64", False)])
def test_swept_batch_equals_stage_launches(dtype, kahan, monkeypatch):
    """Instances from 8 to 254 unknowns per side with every mix of boundary kinds; odd and even
    step counts (the state ends in the caller's array either way)."""
    rng = np.random.default_rng(11)
    lows, dts = [], []
    for n in (10, 11, 33, 65, 66, 67, 100, 122, 123, 180, 256):
        bc = tuple(int(b) for b in rng.integers(0, 2, 4))
        lows.append(lower(*systems.diffreact2d(n, 0.05, 1.0 + 0.1 * n, bc, dtype=dtype)))
        dts.append(2.0 / (n - 1) ** 2)
    batch = BatchProblem(lows)
    monkeypatch.setenv("MOL_SWEEP", "0")
    stage = BatchProblem(lows)
    u0 = rng.uniform(0.1, 0.9, batch.n_unknowns)
    tol = 1e-13 if dtype == "f64" else 4 * 2.0 ** -24 * (1 if kahan else 4)
    for N in (1, 4):
        print("  sweep batch %s kahan=%s N=%d" % (dtype, kahan, N), flush=True)
        got = _run(batch, u0, 0.0, min(dts), N, kahan=kahan)
        ref = _run(stage, u0, 0.0, min(dts), N, kahan=kahan)
        assert np.max(np.abs(got - ref)) <= tol


@pytest.mark.parametrize("dtype,kahan", [("f32", True), ("f32", False), ("f64", True), ("f64", False)])
@pytest.mark.parametrize("first", [0, 1, 2])
def test_mixed_periodic_batch_equals_stage_launches(first, dtype, kahan, monkeypatch):
    """Periodic, non-periodic and one-axis-periodic instances in one batch, each kind first, at the
    column counts where the two kinds differ in windows; the workspace holds NaN before the run."""
    rng = np.random.default_rng(5)
    kinds = [(True, True), (False, False), (True, False), (False, True)]
    sizes = [(c, 12 + c // 4, *kinds[(j + first) % 4]) for c in (57, 64, 112, 120) for j in range(4)]
    lows = [lower(*axis_system(c + (1 if xp else 2), r + (1 if yp else 2), xp, yp, dtype)) for c, r, xp, yp in sizes]
    batch = BatchProblem(lows)
    monkeypatch.setenv("MOL_SWEEP", "0")
    stage = BatchProblem(lows)
    # a run from NaN leaves NaN in every vector of the batch's workspace that a step writes
    _run(batch, np.full(batch.n_unknowns, np.nan), 0.0, 1e-5, 3, kahan=kahan)
    u0 = rng.uniform(0.1, 0.9, batch.n_unknowns)
    tol = 1e-13 if dtype == "f64" else 4 * 2.0 ** -24 * (1 if kahan else 4)
    for N in (1, 4):
        print("  mixed batch first=%d %s kahan=%s N=%d" % (first, dtype, kahan, N), flush=True)
        got = _run(batch, u0, 0.0, 1e-4, N, kahan=kahan)
        ref = _run(stage, u0, 0.0, 1e-4, N, kahan=kahan)
        assert np.all(np.isfinite(got))
        assert np.max(np.abs(got - ref)) <= tol


@pytest.mark.parametrize("kahan", [False, True])
@pytest.mark.parametrize("nx,ny,rows", [(9, 30, 4), (57, 33, 7), (64, 20, 5), (120, 64, 64), (121, 40, 9)])
@pytest.mark.parametrize("xper,yper", [(True, False), (False, True)])
def test_swept_steps_with_one_periodic_axis(xper, yper, nx, ny, rows, kahan, monkeypatch):
    monkeypatch.setenv("MOL_SWEEP", "1")
    monkeypatch.setenv("MOL_SWEEP_ROWS", str(rows))
    prob = molgpu.ODEProblem(lower(*axis_system(nx + (1 if xper else 2), ny + (1 if yper else 2), xper, yper)))
    u0 = np.random.default_rng(nx).uniform(0.1, 0.9, prob.lowered.n_unknowns)
    print("  sweep per=(%s, %s) %dx%d rows=%d kahan=%s" % (xper, yper, nx, ny, rows, kahan), flush=True)
    ref = _run(prob, u0, 0.0, 1e-5, 5, kahan=kahan, fused=False)
    got = _run(prob, u0, 0.0, 1e-5, 5, kahan=kahan)
    assert np.max(np.abs(got - ref)) <= 1e-13 * (1 + np.max(np.abs(ref)))


# systems whose plain step runs on tiles and whose compensated step is swept (199^2), both swept, and
# eight FP64 variables, whose sweep keeps part of its rows in scratch memory
@pytest.mark.parametrize("nf,dtype,n", [(3, "f64", 200), (4, "f32", 200), (3, "f64", 364), (8, "f64", 200), (8, "f64", 364)])
@pytest.mark.parametrize("periodic", [True, False])
def test_steps_of_many_variables_equal_stage_launches(nf, dtype, n, periodic):
    prob = molgpu.ODEProblem(lower(*coupled_system(nf, n, periodic, dtype)))
    u0 = np.random.default_rng(n).uniform(0.1, 0.9, prob.lowered.n_unknowns)
    dt = 0.5 / n ** 2
    eps = 1e-13 if dtype == "f64" else 16 * 2.0 ** -24
    for kahan in (False, True):
        print("  many variables nf=%d %s n=%d kahan=%s" % (nf, dtype, n, kahan), flush=True)
        ref = _run(prob, u0, 0.0, dt, 5, kahan=kahan, fused=False)
        got = _run(prob, u0, 0.0, dt, 5, kahan=kahan)
        assert np.max(np.abs(got - ref)) <= eps * (1 + np.max(np.abs(ref)))


def _advected(nx, ny, left, dtype="f64"):
    """u_t = -u_x - u_y, upwind: a node reads itself and the nodes below it on either axis."""
    t, x, y = parameters("t x y")
    u = variables("u")
    Dx, Dy = Differential(x), Differential(y)
    U = u(t, x, y)
    bcs = [Eq(u(0, x, y), 0.5), Eq(u(t, 0, y), 0.2) if left == 0 else Eq(Dx(u(t, 0, y)), 0), Eq(u(t, 1, y), 0.1),
           Eq(u(t, x, 0), 0.3), Eq(u(t, x, 1), 0.4)]
    return lower(PDESystem([Eq(Differential(t)(U), -Dx(U) - Dy(U))], bcs, [Interval(v, 0.0, 1.0) for v in (t, x, y)],
                           [t, x, y], [U]), MOLFiniteDifference({x: nx, y: ny}, t, advection_scheme=UpwindScheme(1), dtype=dtype))


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["upwind", "centred"])
def test_batch_sides_with_a_value_do_not_read_the_nodes_next_to_them(kind, bad, dtype, monkeypatch):
    """One infinite or undefined node, the second from each side that has a value: it spreads
    where the stencil carries it, as with stage launches, and not through the side's ghost."""
    if kind == "upwind":
        lows = [_advected(30, 25, 0, dtype), _advected(80, 20, 1, dtype), _advected(70, 40, 0, dtype)]
    else:
        lows = [lower(*systems.diffreact2d(n, 0.05, 1.0, bc, dtype=dtype)) for n, bc in
                ((30, (0, 0, 0, 0)), (80, (0, 1, 1, 0)), (70, (1, 0, 0, 1)))]
    batch = BatchProblem(lows)
    monkeypatch.setenv("MOL_SWEEP", "0")
    stage = BatchProblem(lows)
    u0 = np.random.default_rng(2).uniform(0.1, 0.9, batch.n_unknowns)
    for low, at in zip(lows, batch.offsets):
        nx, ny = (int(n) - 2 for n in low.n[:2])
        v = u0[at:at + nx * ny].reshape(ny, nx)
        v[ny // 2, 1] = v[1, nx // 2] = bad
    for kahan in (False, True):
        print("  batch sides %s %s %s kahan=%s" % (kind, bad, dtype, kahan), flush=True)
        got = _run(batch, u0, 0.0, 1e-4, 1, kahan=kahan)
        ref = _run(stage, u0, 0.0, 1e-4, 1, kahan=kahan)
        assert np.isfinite(ref).sum() > 0.5 * ref.size
        np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))
        ok = np.isfinite(ref)
        assert np.max(np.abs(got[ok] - ref[ok])) <= (1e-13 if dtype == "f64" else 16 * 2.0 ** -24)
