"""3D divergence form marched along z: the generated forward and reverse-mode kernels on the CPU
against the tile kernels of the same system, over boundary kinds, coefficients, tiles and chunks."""
import os
import sys

import numpy as np
import pytest
import sympy as sp

import oracle as orc
from molgpu import systems
from molgpu.discretization import MOLFiniteDifference, lower
from molgpu.pdesys import Differential, Eq, Interval, PDESystem, grid_field, parameters, variables

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "genhost"))
import genhost  # noqa: E402

t, x, y, z, k0 = parameters("t x y z k0")
u = variables("u")
D = {v: Differential(v) for v in (t, x, y, z)}
U = u(t, x, y, z)


def system(coef, extra, bcs, n=(13, 21, 27), params=None, **opt):
    """u_t = sum over the axes of d/dx(coef[axis] du/dx) + extra; boundary equations per side."""
    eq = Eq(D[t](U), sum(D[v](a * D[v](U)) for v, a in zip((x, y, z), coef)) + extra)
    sys_ = PDESystem([eq], [Eq(u(0, x, y, z), 0)] + bcs, [Interval(v, 0.0, 1.0) for v in (t, x, y, z)], [t, x, y, z],
                     [U], **({"ps": params} if params else {}))
    return lower(sys_, MOLFiniteDifference(dict(zip((x, y, z), n)), t, **opt))


def side(v, b):
    args = [t, x, y, z]
    args[1 + (x, y, z).index(v)] = b
    return u(*args), D[v](u(*args))


def neumann():
    return [Eq(side(v, b)[1], 0) for v in (x, y, z) for b in (0, 1)]


def mixed():
    """Dirichlet varying along the side and in time, Neumann with a value, Robin."""
    (xl, dxl), (xh, dxh), (yl, dyl), (yh, dyh) = side(x, 0), side(x, 1), side(y, 0), side(y, 1)
    (zl, dzl), (zh, dzh) = side(z, 0), side(z, 1)
    return [Eq(xl, sp.sin(3 * t) * y + z), Eq(dxh, sp.cos(2 * y)), Eq(dyl, 0.3), Eq(yh + 0.5 * dyh, x * z),
            Eq(2 * zl - dzl, t), Eq(zh, x * y)]


d0, s0, w0 = grid_field("d0"), grid_field("s0"), grid_field("w0")
F = (x, y, z)
SYSTEMS = {
    "fields": lambda: system([d0(*F) * (1 + U ** 2)] * 3, s0(*F), neumann()),
    "mixed": lambda: system([d0(*F) * (1 + U ** 2), d0(*F) + s0(*F), sp.exp(-U) * (2 + sp.sin(t))], w0(*F) * U ** 2 - U,
                            mixed()),
    "no_fields": lambda: system([1 + U ** 2, 2 + U, 1 + U], sp.sin(3 * x) * y * U, mixed(), n=(12, 12, 14)),
    "scaled": lambda: system([-(1 + U ** 2), -(1 + U ** 2), -(3 + U)], 0, neumann(), n=(34, 12, 13)),
}


@pytest.mark.parametrize("tile", ["32,8,8", "8,8,4", "16,16,64"])
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_march_equals_tiles(name, tile, monkeypatch):
    import molgpu
    low = SYSTEMS[name]()
    rng = np.random.default_rng(len(name))
    v = rng.uniform(-0.8, 0.8, low.n_unknowns)
    lam = rng.standard_normal(low.n_unknowns)
    aux = {a: rng.uniform(0.5, 1.5, low.n) for a in low.aux}
    monkeypatch.setenv("MOL_FLUX", "0")
    ref = genhost.rhs(low, v, t=0.4, aux=aux)
    rl, rg = genhost.vjp(low, v, lam, t=0.4, aux=aux)
    monkeypatch.setenv("MOL_FLUX", "1")
    monkeypatch.setenv("MOL_FLUX_TILE", tile)
    monkeypatch.setenv("MOL_FLUX_VJP_TILE", tile)
    assert "mol_flux_rhs<" in molgpu.codegen(low) and "mol_flux_vjp<" in molgpu.codegen(low, vjp=True)
    got = genhost.rhs(low, v, t=0.4, aux=aux)
    gl, gg = genhost.vjp(low, v, lam, t=0.4, aux=aux)
    # some fifty roundings of terms of the size of the largest result
    assert np.max(np.abs(got - ref)) <= 1e-13 * np.max(np.abs(ref))
    assert np.max(np.abs(gl - rl)) <= 1e-13 * np.max(np.abs(rl))
    if low.aux:
        for a in range(len(low.aux)):
            assert np.max(np.abs(gg[a] - rg[a])) <= 1e-13 * np.max(np.abs(rg[a])), low.aux[a]


def test_march_against_oracle(monkeypatch):
    monkeypatch.setenv("MOL_FLUX", "1")
    n = 19
    low = lower(*systems.nonlindiff3d(n=n))
    f0 = 0.5 + 0.5 * np.abs(systems.gaussian_field3d(n, 1))
    src = systems.gaussian_field3d(n, 2)
    v = np.random.default_rng(6).uniform(-1, 1, low.n_unknowns)
    ref = orc.nonlindiff3d_rhs(n, f0.reshape(-1, order="F"), src.reshape(-1, order="F"), v)
    got = genhost.rhs(low, v, aux={"d0": f0, "s": src})
    assert np.max(np.abs(got - ref)) <= 1e-13 * np.max(np.abs(ref))


@pytest.mark.parametrize("name", ["short", "order4", "advection", "slot_product", "node_coordinate", "tile"])
def test_other_systems_keep_the_tiles(name, monkeypatch):
    import molgpu
    monkeypatch.setenv("MOL_FLUX", "1")
    a = [1 + U ** 2] * 3
    low, tile = {
        "short": lambda: (system(a, 0, neumann(), n=(11, 20, 20)), None),
        "order4": lambda: (system(a, 0, neumann(), n=(21, 21, 21), approx_order=4), None),
        "advection": lambda: (system(a, D[x](U), neumann()), None),
        "slot_product": lambda: (system([U * (1 + U)] * 3, (D[x]((1 + U) * D[x](U))) * U, neumann()), None),
        "node_coordinate": lambda: (system([1 + x * U] * 3, 0, neumann()), None),
        "tile": lambda: (system(a, 0, neumann()), (8, 4, 4)),
    }[name]()
    for vjp in (False, True):
        assert "mol_flux_" not in molgpu.codegen(low, tile=tile, vjp=vjp).split("#include")[1].split("struct GeoB")[-1]


@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_march_compiles_for_gfx950(name, monkeypatch):
    import molgpu
    monkeypatch.setenv("MOL_FLUX", "1")
    for vjp in (False, True):
        assert "mol_flux_" in molgpu.codegen(SYSTEMS[name](), vjp=vjp, compile=True)


def test_sizes_that_the_march_takes():
    """Right-hand sides from 48^3 unknowns, with two interpolated fields from 50^3 (at 48^3 tiles are as
    fast or faster)."""
    import molgpu
    one, two = [d0(*F) * (1 + U ** 2)] * 3, [d0(*F) * (1 + U ** 2), d0(*F) + s0(*F), 1 + U]
    for coef, least in ((one, 50), (two, 52)):
        for n in (least - 1, least):
            src = molgpu.codegen(system(coef, 0, neumann(), n=(n, n, n)))
            assert ("mol_flux_rhs<GeoB>(" in src) == (n >= least)
