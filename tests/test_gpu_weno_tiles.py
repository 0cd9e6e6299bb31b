"""GPU: tile heights and nodes per thread that the size rules choose for reach-two 2D stencils,
against small tiles of the same system."""
import numpy as np
import pytest

import molgpu
from molgpu import Differential, Eq, Interval, MOLFiniteDifference, PDESystem, WENOScheme, parameters, variables

pytestmark = pytest.mark.gpu


def _burgers(nx, ny, dtype):
    t, x, y = parameters("t x y")
    u = variables("u")
    U = u(t, x, y)
    eq = Eq(Differential(t)(U), -U * Differential(x)(U) - U * Differential(y)(U))
    bcs = [Eq(u(0, x, y), 0.5), Eq(u(t, 0, y), u(t, 1, y)), Eq(u(t, x, 0), u(t, x, 1))]
    return molgpu.discretize(PDESystem([eq], bcs, [Interval(v, 0.0, 1.0) for v in (t, x, y)], [t, x, y], [U]),
                             MOLFiniteDifference({x: nx + 1, y: ny + 1}, t, advection_scheme=WENOScheme(1e-6), dtype=dtype))


# whole tiles; cut along either axis; 12, 20 and 28 rows per tile
@pytest.mark.parametrize("nx,ny", [(1024, 1024), (1024, 1030), (1029, 1024), (1447, 1447), (1300, 1300), (1700, 1500)])
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_chosen_tiles_equal_small_tiles(nx, ny, dtype):
    import torch
    prob = _burgers(nx, ny, dtype)
    td = prob.torch_dtype()
    u = torch.tensor(np.random.default_rng(nx).uniform(0.2, 1.2, nx * ny), device="cuda").to(td)
    got, ref = torch.empty_like(u), torch.empty_like(u)
    print("  weno tiles %dx%d %s" % (nx, ny, dtype), flush=True)
    prob.f(got, u, None, 0.0)
    small = _burgers(nx, ny, dtype)
    small.set_tile(32, 8, 1)
    small.f(ref, u, None, 0.0)
    torch.cuda.synchronize()
    # the same arithmetic per node, contracted differently at most: a few roundings of u du/dx
    tol = (1e-14 if dtype == "f64" else 4e-6) * max(nx, ny)
    assert float((got - ref).abs().max()) <= tol
