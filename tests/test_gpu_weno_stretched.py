"""GPU: WENO5 on stretched nodes along both axes (coefficient columns of the tile in LDS along x,
scalar rows along y) at the sizes where tiles are ragged, wider than the table in LDS or cut by the
ends, line by line against the derivative in extended precision and, next to the ends, the oracle."""
import numpy as np
import pytest

import oracle as orc
import molgpu
from molgpu import systems
from molgpu.discretization import MOLFiniteDifference, WENOScheme, lower
from molgpu.pdesys import Differential, Eq, Interval, PDESystem, parameters, variables
from test_weno_nonuniform import exact_derivative

pytestmark = pytest.mark.gpu
C = (1.0, 0.5)


def _nodes(n, seed):
    h = 1.0 + 0.3 * (2 * np.random.default_rng(seed).random(n - 1) - 1)
    x = np.concatenate([[0.0], np.cumsum(h)]) / h.sum()
    x[-1] = 1.0
    return x


def _problem(nx, ny, periodic, dtype="f64"):
    t, x, y = parameters("t x y")
    u = variables("u")
    U = u(t, x, y)
    eq = Eq(Differential(t)(U), -C[0] * Differential(x)(U) - C[1] * Differential(y)(U))
    if periodic:
        bcs = [Eq(u(0, x, y), 0.5), Eq(u(t, 0, y), u(t, 1, y)), Eq(u(t, x, 0), u(t, x, 1))]
    else:
        bcs = [Eq(u(0, x, y), 0.5), Eq(u(t, 0, y), 0.25), Eq(u(t, 1, y), 0.375), Eq(u(t, x, 0), 0.125),
               Eq(u(t, x, 1), 0.5)]
    nodes = [_nodes(nx, 3), _nodes(ny, 4)]
    low = lower(PDESystem([eq], bcs, [Interval(v, 0.0, 1.0) for v in (t, x, y)], [t, x, y], [U]),
                MOLFiniteDifference({x: nodes[0], y: nodes[1]}, t, advection_scheme=WENOScheme(1e-6), dtype=dtype))
    return molgpu.ODEProblem(low), nodes


def _reference(nodes, periodic, v):
    """Extended precision where the target is centred; next to an end the oracle's one-sided targets
    on distances to the node (exact differences, so that the oracle does not round whole coordinates)."""
    out = []
    for x, c, ends, w in ((nodes[0], C[0], (0.25, 0.375), v), (nodes[1], C[1], (0.125, 0.5), v.T)):
        if periodic:
            d = exact_derivative(x, w, True)
        else:
            w = np.concatenate([np.full((len(w), 1), ends[0]), w, np.full((len(w), 1), ends[1])], axis=1)
            d = np.stack([[orc.weno_nu(np.ascontiguousarray(r[:5]), x[:5] - x[1], 1e-6, 2)] +
                          [0.0] * (len(x) - 4) + [orc.weno_nu(np.ascontiguousarray(r[-5:]), x[-5:] - x[-2], 1e-6, 4)]
                          for r in w])
            d[:, 1:-1] = exact_derivative(x, w, False)
        out.append(-c * d)
    return out[0] + out[1].T


# tiles of whole waves, odd ones, wider than 128 nodes (which read the axis table); the default at
# sizes whose last tiles hold one column or one row, and whole ones
@pytest.mark.parametrize("nx,ny,tile", [(151, 38, (64, 8, 1)), (151, 38, (20, 7, 1)), (151, 38, (130, 4, 1)),
                                        (67, 35, None), (131, 514, None), (515, 259, None), (705, 545, None)])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_rhs_on_stretched_nodes_against_oracle(dtype, periodic, nx, ny, tile):
    import torch
    prob, nodes = _problem(nx, ny, periodic, dtype)
    if tile is not None:
        prob.set_tile(*tile)
    low = prob.lowered
    shape = [h - l + 1 for l, h in zip(low.lo[0], low.hi[0])][::-1]
    v = np.random.default_rng(nx).uniform(0.0, 1.0, shape).astype(np.float32).astype(np.float64)
    u = torch.tensor(v.reshape(-1), device="cuda").to(prob.torch_dtype())
    du = torch.empty_like(u)
    print("  stretched %s periodic=%s %dx%d tile=%s" % (dtype, periodic, nx, ny, tile), flush=True)
    prob.f(du, u, None, 0.0)
    got = du.double().cpu().numpy().reshape(shape)
    # differences of values up to one over the shortest spacings, weights from sums of their squares
    eps = 2.0 ** -53 if dtype == "f64" else 2.0 ** -24
    tol = 64 * eps * sum(c / np.diff(x).min() for c, x in zip(C, nodes))
    assert np.max(np.abs(got - _reference(nodes, periodic, v))) <= tol


@pytest.mark.parametrize("nx,ny", [(40, 33), (200, 131)])
def test_fused_steps_on_stretched_periodic_nodes_equal_stage_launches(nx, ny):
    import torch
    prob, nodes = _problem(nx, ny, True)
    v = np.random.default_rng(1).uniform(0.0, 1.0, prob.lowered.n_unknowns)
    out = []
    for fused in (True, False):
        u = torch.tensor(v, device="cuda")
        print("  stretched rk4 %dx%d fused=%s" % (nx, ny, fused), flush=True)
        prob.integrate(u, 0.0, 0.1 * np.diff(nodes[0]).min(), 5, molgpu.RK4, fused=fused)
        out.append(u.cpu().numpy())
    assert prob.plan()["fused_tiles"] > 0
    assert np.max(np.abs(out[0] - out[1])) <= 1e-12 * (1 + np.max(np.abs(out[1])))
