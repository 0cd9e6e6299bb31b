"""Reverse mode of WENO5 systems whose tile kernel takes more registers than a work-group of 1024
threads leaves it: such a kernel is never launched (the queue would refuse it and end the process),
it is built with fewer threads."""
import numpy as np
import pytest

import molgpu
from molgpu.discretization import MOLFiniteDifference, WENOScheme, lower
from molgpu.pdesys import Differential, Eq, Interval, PDESystem, parameters, variables


def coupled_burgers(nf, n, periodic, stretched, dtype):
    """u_t = -u u_x - v u_y, and so on around nf variables."""
    t, x, y = parameters("t x y")
    vs = [variables("u%d" % k) for k in range(nf)]
    U = [v(t, x, y) for v in vs]
    D = Differential
    eqs = [Eq(D(t)(U[k]), -U[k] * D(x)(U[k]) - U[(k + 1) % nf] * D(y)(U[k])) for k in range(nf)]
    bcs = []
    for v in vs:
        bcs.append(Eq(v(0, x, y), 0.5))
        for args in (lambda b: (t, b, y), lambda b: (t, x, b)):
            bcs += [Eq(v(*args(0)), v(*args(1)))] if periodic else [Eq(v(*args(0)), 0.5), Eq(v(*args(1)), 0.4)]
    grid = n
    if stretched:
        h = 1.0 + 0.3 * (2 * np.random.default_rng(7).random(n - 1) - 1)
        grid = np.concatenate([[0.0], np.cumsum(h)]) / h.sum()
        grid[-1] = 1.0
    return lower(PDESystem(eqs, bcs, [Interval(q, 0.0, 1.0) for q in (t, x, y)], [t, x, y], U),
                 MOLFiniteDifference({x: grid, y: grid}, t, advection_scheme=WENOScheme(1e-6), dtype=dtype))


# (136, 130 and 144 registers per lane with 1024 threads, which leave 128)
CASES = [(2, True, False, "f64"), (2, False, True, "f64"), (1, False, True, "f32")]


@pytest.mark.parametrize("nf,periodic,stretched,dtype", CASES)
def test_kernel_is_built_with_threads_that_its_registers_allow(nf, periodic, stretched, dtype):
    low = coupled_burgers(nf, 700, periodic, stretched, dtype)
    assert "__launch_bounds__(1024) mol_vjp_tiles" in molgpu.codegen(low, vjp=True)   # as asked for
    assert "__launch_bounds__(512) mol_vjp_tiles" in molgpu.codegen(low, vjp=True, compile=True)


@pytest.mark.gpu
@pytest.mark.parametrize("nf,periodic,stretched,dtype", CASES)
def test_product_with_large_tiles_equals_small_tiles(nf, periodic, stretched, dtype, monkeypatch):
    """Tiles of 1024 nodes against tiles of 128: the same sums, rounded once more per tile that
    holds a part (four at most, each of up to eleven terms)."""
    import torch
    rng = np.random.default_rng(3)
    got = []
    for tile in ("32,32,1", "16,8,1"):
        monkeypatch.setenv("MOL_VJP_TILE", tile)
        prob = molgpu.ODEProblem(coupled_burgers(nf, 70, periodic, stretched, dtype))
        if not got:
            u, lam = (torch.tensor(rng.uniform(0.2, 1.0, prob.lowered.n_unknowns), device="cuda").to(prob.torch_dtype())
                      for _ in range(2))
        print("  vjp registers %s tile %s" % ((nf, periodic, stretched, dtype), tile), flush=True)
        got.append(prob.vjp(u, lam, 0.0).double().cpu().numpy())
    eps = 2.0 ** -53 if dtype == "f64" else 2.0 ** -24
    assert np.all(np.isfinite(got[0]))
    assert np.max(np.abs(got[0] - got[1])) <= 64 * eps * np.max(np.abs(got[1]))
