"""Where a march or register sweep does not build, the kernels that it stands in for run: tiles for
the right-hand side, its vector-Jacobian product and the fused step, stage launches for batches."""
import numpy as np
import pytest

import molgpu
from molgpu import systems
from molgpu.batch import BatchProblem, codegen_batched
from molgpu.discretization import lower


def _batch(dtype="f32"):
    return [lower(*systems.diffreact2d(n, 0.05, 1.0 + 0.1 * n, (n & 1, 0, 1, 0), dtype=dtype)) for n in (20, 33, 70)]


@pytest.mark.parametrize("vjp", [False, True])
def test_march_that_does_not_build_leaves_the_tiles(vjp, monkeypatch):
    low = lower(*systems.nonlindiff3d(n=60))
    assert "mol_flux_" in molgpu.codegen(low, vjp=vjp, compile=True)
    monkeypatch.setenv("MOL_JIT_FAIL", "mol_flux_")
    src = molgpu.codegen(low, vjp=vjp, compile=True)
    monkeypatch.delenv("MOL_JIT_FAIL")
    monkeypatch.setenv("MOL_FLUX", "0")
    assert src == molgpu.codegen(low, vjp=vjp, compile=True)


def test_sweep_that_does_not_build_leaves_the_tiles(monkeypatch):
    low = lower(*systems.diffreact2d(90, 0.1, 2.0, (0, 1, 1, 0)))
    assert "mol_rk4_sweep<" in molgpu.codegen(low, fused=True, compile=True)
    monkeypatch.setenv("MOL_JIT_FAIL", "mol_rk4_sweep<")
    src = molgpu.codegen(low, fused=True, compile=True)
    assert "mol_rk4_sweep<" not in src and "mol_rk4_fused_tile<" in src


def test_batch_whose_step_does_not_build_keeps_its_stages(monkeypatch):
    assert "mol_batch_rk4" in codegen_batched(_batch(), compile=True)
    monkeypatch.setenv("MOL_JIT_FAIL", "mol_rk4_sweep<")
    src = codegen_batched(_batch(), compile=True)
    assert "mol_batch_rk4" not in src and "mol_batch_tiles" in src


@pytest.mark.gpu
def test_results_of_what_runs_instead(monkeypatch):
    """The same results as with the march and the sweep switched off."""
    import torch

    def run(env):
        for k in ("MOL_JIT_FAIL", "MOL_FLUX", "MOL_SWEEP"):
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        print("  fallback %s" % env, flush=True)
        out = []
        prob = molgpu.discretize(*systems.nonlindiff3d(n=52))
        for a in prob.lowered.aux:
            prob.set_grid_field(a, torch.linspace(0.5, 1.5, 52 ** 3, dtype=torch.float64, device="cuda"))
        u = torch.linspace(-0.5, 0.5, prob.lowered.n_unknowns, dtype=torch.float64, device="cuda")
        du = torch.empty_like(u)
        prob.f(du, u, None, 0.0)
        out += [du, prob.vjp(u, du, 0.0)]
        for b in (molgpu.discretize(*systems.diffreact2d(300, 0.1, 2.0, (0, 1, 1, 0))), BatchProblem(_batch())):
            n = b.lowered.n_unknowns if isinstance(b, molgpu.ODEProblem) else b.n_unknowns
            for kahan in (False, True):
                v = torch.linspace(0.1, 0.9, n, dtype=torch.float64, device="cuda").to(b.torch_dtype())
                b.integrate(v, 0.0, 1e-6, 3, molgpu.RK4, kahan=kahan)
                out.append(v)
        return [o.cpu().numpy() for o in out]

    def same(got, ref):
        # (index 1, the product: sums by atomics, in any order, of up to 26 terms)
        for k, (a, b) in enumerate(zip(got, ref)):
            assert np.max(np.abs(a - b)) <= (64 * 2.0 ** -53 * np.max(np.abs(b)) if k == 1 else 0.0)

    off = run({"MOL_FLUX": "0", "MOL_SWEEP": "0"})
    same(run({"MOL_JIT_FAIL": "mol_flux_"})[:2], off[:2])
    same(run({"MOL_JIT_FAIL": "mol_rk4_sweep<", "MOL_FLUX": "0"}), off)
