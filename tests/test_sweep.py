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


def axis_system(nx, ny, xper, yper, dtype="f64", k=1.0):
    """u_t = 0.05 (u_xx + u_yy) + k u (1 - u), each axis periodic or from a value to a flux."""
    t, x, y = parameters("t x y")
    u = variables("u")
    Dx, Dy = Differential(x), Differential(y)
    U = u(t, x, y)
    eq = Eq(Differential(t)(U), 0.05 * ((Dx ** 2)(U) + (Dy ** 2)(U)) + k * U * (1 - U))
    bcs = [Eq(u(0, x, y), 0.5)]
    bcs += [Eq(u(t, 0, y), u(t, 1, y))] if xper else [Eq(u(t, 0, y), 0.2), Eq(Dx(u(t, 1, y)), 0.1)]
    bcs += [Eq(u(t, x, 0), u(t, x, 1))] if yper else [Eq(Dy(u(t, x, 0)), 0.3), Eq(u(t, x, 1), 0.4)]
    return PDESystem([eq], bcs, [Interval(v, 0.0, 1.0) for v in (t, x, y)], [t, x, y], [U]), \
        MOLFiniteDifference({x: nx, y: ny}, t, dtype=dtype)


@pytest.mark.parametrize("xper,yper", [(True, False), (False, True)])
@pytest.mark.parametrize("rows", [4, 9, 64])
def test_swept_step_with_one_periodic_axis(xper, yper, rows, monkeypatch):
    import molgpu
    monkeypatch.setenv("MOL_SWEEP", "1")
    monkeypatch.setenv("MOL_SWEEP_ROWS", str(rows))
    low = lower(*axis_system(23, 31, xper, yper))
    assert "mol_rk4_sweep<" in molgpu.codegen(low, fused=True)
    w = np.random.default_rng(rows).uniform(0.1, 0.9, low.n_unknowns)
    got, _ = genhost.rk4_fused(low, w, 0.0, 1e-3)
    ref = _rk4(lambda v, s: genhost.rhs(low, v, t=s), w, 0.0, 1e-3)
    assert np.max(np.abs(got - ref)) <= 1e-14 * (1 + np.max(np.abs(ref)))


# columns around the edges of one and two windows, periodic and not
MIXED = [(n, 20, xper, yper) for n in (9, 56, 57, 63, 64, 65, 112, 113, 119, 120, 121) for xper, yper in
         ((True, True), (False, False), (True, False), (False, True))]


@pytest.mark.parametrize("first", [0, 1])
def test_waves_of_a_mixed_batch_own_every_node_once(first, monkeypatch):
    """Periodic and non-periodic instances in one batch, either kind first: the columns and rows
    that the waves of an instance own tile it, each inside the part of its window that four
    stages leave valid."""
    from molgpu.batch import codegen_batched
    monkeypatch.setenv("MOL_SWEEP_ROWS", "7")
    order = MIXED[first:] + MIXED[:first]
    lows = [lower(*axis_system(c + (1 if xp else 2), r + (1 if yp else 2), xp, yp, "f32")) for c, r, xp, yp in order]
    waves = [[int(v) for v in ln.split()] for ln in codegen_batched(lows, waves=True).splitlines()]
    own = [np.zeros((c, r), dtype=int) for c, r, _, _ in order]
    for i, _, xb, x0, x1, y0, y1, _ in waves:
        c, r, xper, yper = order[i]
        assert 0 <= x0 < x1 <= c and 0 <= y0 < y1 <= r and (y0 == 0 or yper or y0 >= 4), (order[i], xb, x0, x1, y0, y1)
        assert xper or xb >= 0, (order[i], xb)
        assert x0 >= xb + 4 or (not xper and x0 == xb == 0), (order[i], xb, x0, x1)
        assert x1 <= xb + 60 or (not xper and x1 == c <= xb + 64), (order[i], xb, x0, x1)
        own[i][x0:x1, y0:y1] += 1
    for i, m in enumerate(own):
        assert np.all(m == 1), (order[i], m.min(), m.max())


def coupled_system(nf, n, periodic, dtype="f64"):
    """u_t = (0.05 + 0.01 k) (u_xx + u_yy) + u (1 - v), and so on around nf variables."""
    t, x, y = parameters("t x y")
    vs = [variables("u%d" % k) for k in range(nf)]
    Dx, Dy = Differential(x), Differential(y)
    U = [v(t, x, y) for v in vs]
    eqs, bcs = [], []
    for k, v in enumerate(vs):
        eqs.append(Eq(Differential(t)(U[k]), (0.05 + 0.01 * k) * ((Dx ** 2)(U[k]) + (Dy ** 2)(U[k])) +
                      U[k] * (1 - U[(k + 1) % nf])))
        bcs.append(Eq(v(0, x, y), 0.5))
        if periodic:
            bcs += [Eq(v(t, 0, y), v(t, 1, y)), Eq(v(t, x, 0), v(t, x, 1))]
        else:
            bcs += [Eq(v(t, 0, y), 0.2), Eq(Dx(v(t, 1, y)), 0), Eq(Dy(v(t, x, 0)), 0), Eq(v(t, x, 1), 0.4)]
    return PDESystem(eqs, bcs, [Interval(q, 0.0, 1.0) for q in (t, x, y)], [t, x, y], U), \
        MOLFiniteDifference({x: n, y: n}, t, dtype=dtype)


# (variables, type, both axes periodic, nodes per side swept from or None for every size)
@pytest.mark.parametrize("nf,dtype,periodic,line", [
    (1, "f64", True, None), (2, "f64", True, None), (3, "f64", True, 363), (7, "f64", True, 363),
    (8, "f64", True, 548), (8, "f64", False, 256), (7, "f64", False, None), (3, "f32", True, 512),
    (8, "f32", True, 512), (8, "f32", False, None)])
def test_sizes_that_the_sweep_takes_by_number_of_variables(nf, dtype, periodic, line):
    """Systems whose tiles are faster on small grids (many variables, periodic axes) keep them."""
    import molgpu
    for side in ([200] if line is None else [line - 1, line]):
        low = lower(*coupled_system(nf, side + (1 if periodic else 2), periodic, dtype))
        assert ("mol_rk4_sweep<" in molgpu.codegen(low, fused=True)) == (line is None or side >= line)


def test_one_sided_operators_keep_boundary_kinds_apart():
    """A class of batched instances serves sides of any kind by zero factors only where the node next
    to a side reads the nodes that the factors stand for; upwind operators get a class per kind."""
    from molgpu.batch import codegen_batched
    from molgpu.discretization import UpwindScheme
    t, x, y = parameters("t x y")
    u = variables("u")
    Dx, Dy = Differential(x), Differential(y)
    U = u(t, x, y)

    def low(left, rhs, **kw):
        bcs = [Eq(u(0, x, y), 0.5), Eq(u(t, 0, y), 0) if left == 0 else Eq(Dx(u(t, 0, y)), 0), Eq(u(t, 1, y), 0),
               Eq(u(t, x, 0), 0), Eq(u(t, x, 1), 0)]
        return lower(PDESystem([Eq(Differential(t)(U), rhs)], bcs, [Interval(v, 0.0, 1.0) for v in (t, x, y)], [t, x, y],
                               [U]), MOLFiniteDifference({x: 30, y: 25}, t, **kw))

    for rhs, kw, classes in ((-Dx(U) - Dy(U), {"advection_scheme": UpwindScheme(1)}, 2),
                             ((Dx ** 2)(U) + (Dy ** 2)(U), {}, 1)):
        src = codegen_batched([low(0, rhs, **kw), low(1, rhs, **kw)], compile=True)
        assert src.count("struct SwpY") == classes


def test_every_instance_of_a_class_is_asked_whether_it_can_be_swept():
    """Two variables on unequal boxes step by stage launches, also behind an instance of the same
    class (boxes are numbers of the instance, not of the class) whose boxes are equal."""
    import copy
    from molgpu.batch import codegen_batched
    low = lower(*coupled_system(2, 30, False))
    other = copy.deepcopy(low)
    other.hi[1][0] -= 1
    assert "mol_rk4_sweep<" in codegen_batched([low, low])
    for order in ([low, other], [other, low]):
        src = codegen_batched(order)
        assert "2 instances, 1 classes" in src and "mol_rk4_sweep<" not in src
