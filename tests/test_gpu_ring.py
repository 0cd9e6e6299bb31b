"""GPU: resident RK4 steps of small 1D systems (the state in registers, lanes exchanging end
nodes by DPP, waves through LDS once per step) at the sizes where the split changes."""
import numpy as np
import pytest

import oracle as orc
import molgpu
from molgpu import systems
from molgpu.discretization import MOLFiniteDifference
from molgpu.pdesys import Differential, Eq, Interval, PDESystem, parameters, variables

pytestmark = pytest.mark.gpu


def _two_fields(n):
    """u_t = u_xx - u v, v_t = v_xx / 2 + u v; u: Dirichlet and Neumann, v: Robin and Dirichlet."""
    t, x = parameters("t x")
    u, v = variables("u v")
    Dx = Differential(x)
    U, V = u(t, x), v(t, x)
    eqs = [Eq(Differential(t)(U), (Dx ** 2)(U) - U * V), Eq(Differential(t)(V), 0.5 * (Dx ** 2)(V) + U * V)]
    bcs = [Eq(u(0, x), x * (1 - x)), Eq(v(0, x), 1 + x), Eq(u(t, 0), 0.2), Eq(Dx(u(t, 1)), 0),
           Eq(v(t, 0) + Dx(v(t, 0)), 1), Eq(v(t, 1), 2)]
    return PDESystem(eqs, bcs, [Interval(t, 0.0, 1.0), Interval(x, 0.0, 1.0)], [t, x], [U, V]), \
        MOLFiniteDifference({x: n}, t)


def _run(prob, u0, dt, N, fused=True):
    import torch
    u = torch.tensor(u0, dtype=prob.torch_dtype(), device="cuda")
    prob.integrate(u, 0.0, dt, N, molgpu.RK4, fused=fused)
    torch.cuda.synchronize()
    return u.cpu().numpy().astype(np.float64)


# unknowns: below one lane's share, whole lanes, one value more, the last one-wave size, the
# first four-wave size, an uneven last wave, the largest resident system
@pytest.mark.parametrize("unknowns", [6, 64, 65, 320, 321, 637, 1024])
@pytest.mark.parametrize("bcl,bch", [((1.0, 0.0, 0.3), (0.0, 1.0, -0.2)), ((1.0, 2.0, 0.1), (2.0, -1.0, 0.4))])
def test_resident_steps_against_oracle(unknowns, bcl, bch):
    n = unknowns + 2
    prob = molgpu.discretize(*systems.heat1d(n=n, D=1.0, bcl=bcl, bch=bch))
    assert prob.plan()["fused_tiles"] == 1
    u0 = np.random.default_rng(unknowns).uniform(-1, 1, unknowns)
    dt, N = 0.3 / (n - 1) ** 2, 23
    print("  ring n=%d %s %s" % (n, bcl, bch), flush=True)
    ref = orc.diffusion1d_integrate(n, 1.0, bcl, bch, u0, 0.0, dt, N)
    assert np.max(np.abs(_run(prob, u0, dt, N) - ref)) <= 1e-13 * (1 + np.max(np.abs(ref)))


@pytest.mark.parametrize("case,n", [("periodic", 24), ("periodic", 81), ("periodic", 321), ("periodic", 322),
                                    ("periodic", 1025), ("two", 24), ("two", 162), ("two", 163), ("two", 700)])
def test_resident_steps_equal_stage_launches(case, n):
    """Reach two on a periodic ring; two variables with different conditions."""
    if case == "periodic":
        prob = molgpu.discretize(*systems.nonlinlap1d(n, True, 0.0, 0.0, 2))
    else:
        prob = molgpu.discretize(*_two_fields(n))
    assert prob.plan()["fused_tiles"] == 1
    u0 = np.random.default_rng(n).uniform(0.2, 1.0, prob.lowered.n_unknowns)
    dt, N = 0.1 / (n - 1) ** 2, 23
    print("  ring %s n=%d" % (case, n), flush=True)
    ref = _run(prob, u0, dt, N, fused=False)
    assert np.max(np.abs(_run(prob, u0, dt, N) - ref)) <= 1e-13 * (1 + np.max(np.abs(ref)))
