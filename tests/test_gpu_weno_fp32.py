"""GPU: FP32 WENO5 weights over the range of smoothness sums that FP32 states can have."""
import numpy as np
import pytest

import molgpu
from molgpu import systems

pytestmark = pytest.mark.gpu


# sums 4 (eps + beta) from 4e-12 up to 1e36: their squares, or reciprocals of them, leave the
# FP32 range at both ends
@pytest.mark.parametrize("scale,eps", [(1.0, 1e-6), (1e-8, 1e-6), (1e-3, 1e-12), (1e8, 1e-6), (1e18, 1e-6)])
def test_fp32_weno_weights_stay_in_range(scale, eps):
    """Smooth data: the FP32 right-hand side of u_t = -u u_x - u u_y equals the FP64 one from the
    same values.  Each difference is exact to one ulp of u, so a derivative is off by a few
    ulp(u)/dx: 10 * 6e-8 * n / (2 pi) of the derivative's maximum."""
    import torch
    n = 33
    x = np.arange(1, n) / (n - 1.0)
    u = np.float32(scale) * (1.5 + np.sin(2 * np.pi * x)[None, :] * np.cos(2 * np.pi * x)[:, None]).astype(np.float32)
    got = {}
    for dtype, td in (("f32", torch.float32), ("f64", torch.float64)):
        prob = molgpu.discretize(*systems.burgers2d(n=n, eps=eps, dtype=dtype))
        ut = torch.tensor(u.reshape(-1), device="cuda").to(td)
        du = torch.empty_like(ut)
        print("  weno %s scale %g eps %g" % (dtype, scale, eps), flush=True)
        prob.f(du, ut, None, 0.0)
        got[dtype] = (du.double() / ut.double()).cpu().numpy()
    assert np.all(np.isfinite(got["f32"]))
    assert np.max(np.abs(got["f32"] - got["f64"])) <= 10 * 6e-8 * n / (2 * np.pi) * np.max(np.abs(got["f64"]))
