"""RK4 step of 2D systems swept along y in registers: the generated kernel on the CPU (one lane
holding whole rows) against the oracle, over strip lengths and boundary kinds."""
import os
import sys

import numpy as np
import pytest

import oracle as orc
from molgpu import systems
from molgpu.discretization import MOLFiniteDifference, lower
from molgpu.pdesys import Differential, Eq, Interval, PDESystem, parameters, variables

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "genhost"))
import genhost  # noqa: E402


def _rk4(f, u, t, dt):
    k1 = f(u, t)
    k2 = f(u + dt / 2 * k1, t + dt / 2)
    k3 = f(u + dt / 2 * k2, t + dt / 2)
    k4 = f(u + dt * k3, t + dt)
    return u + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)


# strips of the least length, a length that leaves a remainder, one strip for the whole box
@pytest.mark.parametrize("rows", [4, 7, 64])
@pytest.mark.parametrize("case", ["periodic", (0, 1, 1, 0), (1, 0, 0, 1)])
def test_swept_step_against_oracle(case, rows, monkeypatch):
    import molgpu
    monkeypatch.setenv("MOL_SWEEP", "1")
    monkeypatch.setenv("MOL_SWEEP_ROWS", str(rows))
    rng = np.random.default_rng(rows)
    if case == "periodic":
        low = lower(*systems.brusselator2d(n=41))
        u = rng.uniform(0.5, 1.5, low.n_unknowns)
        got, _ = genhost.rk4_fused(low, u, 1.2, 1e-6)
        ref = orc.bruss2d_integrate(41, u, 1.2, 1e-6, 1)
    else:
        low = lower(*systems.diffreact2d(37, 0.1, 2.0, case))
        u = rng.uniform(0.5, 1.5, low.n_unknowns)
        got, _ = genhost.rk4_fused(low, u, 0.0, 1e-4)
        ref = _rk4(lambda w, t: orc.diffreact2d_rhs(37, 0.1, 2.0, case, w, t), u, 0.0, 1e-4)
    assert "mol_rk4_sweep<" in molgpu.codegen(low, fused=True)
    assert np.max(np.abs(got - ref)) <= 1e-14 * np.max(np.abs(ref))


def test_swept_step_with_time_dependent_boundaries(monkeypatch):
    """Boundary values that vary in time and along the side, coordinates in the equation."""
    import molgpu
    import sympy as sp
    t, x, y = parameters("t x y")
    u = variables("u")
    Dx, Dy = Differential(x), Differential(y)
    eq = Eq(Differential(t)(u(t, x, y)), 0.05 * ((Dx ** 2)(u(t, x, y)) + (Dy ** 2)(u(t, x, y))) + sp.sin(3 * x) * y * u(t, x, y))
    bcs = [Eq(u(0, x, y), x * (1 - x) * y), Eq(u(t, 0, y), sp.sin(5 * t) * y), Eq(Dx(u(t, 1, y)), sp.cos(2 * y)),
           Eq(Dy(u(t, x, 0)), x), Eq(u(t, x, 1) + Dy(u(t, x, 1)), sp.cos(3 * t) * x)]
    low = lower(PDESystem([eq], bcs, [Interval(v, 0.0, 1.0) for v in (t, x, y)], [t, x, y], [u(t, x, y)]),
                MOLFiniteDifference({x: 23, y: 31}, t))
    monkeypatch.setenv("MOL_SWEEP", "1")
    monkeypatch.setenv("MOL_SWEEP_ROWS", "9")
    assert "mol_rk4_sweep<" in molgpu.codegen(low, fused=True)
    w = np.random.default_rng(1).uniform(-1, 1, low.n_unknowns)
    got, tn = genhost.rk4_fused(low, w, 0.3, 1e-3)
    ref = _rk4(lambda v, s: genhost.rhs(low, v, t=s), w, 0.3, 1e-3)
    assert tn == 0.3 + 1e-3
    assert np.max(np.abs(got - ref)) <= 1e-13 * (1 + np.max(np.abs(ref)))


def test_systems_that_the_sweep_does_not_hold_keep_the_tile_step(monkeypatch):
    """Reach two and mixed derivatives stay on the tile kernel."""
    import molgpu
    monkeypatch.setenv("MOL_SWEEP", "1")
    assert "mol_rk4_sweep<" not in molgpu.codegen(lower(*systems.brusselator2d(n=65, approx_order=4)), fused=True)
    assert "mol_rk4_sweep<" not in molgpu.codegen(lower(*systems.mixed2d(41, 0.3)), fused=True)
