"""GPU: the launch plan names the kernels that run."""
import pytest

import molgpu
from molgpu import systems
from molgpu.batch import BatchProblem
from molgpu.discretization import lower
from test_sweep import coupled_system

pytestmark = pytest.mark.gpu


def test_plan_of_marched_right_hand_sides():
    import torch
    for n, march in ((40, 0), (64, 1)):
        prob = molgpu.discretize(*systems.nonlindiff3d(n))
        for a in prob.lowered.aux:
            prob.set_grid_field(a, torch.ones(n ** 3, dtype=torch.float64, device="cuda"))
        plan = prob.plan()
        assert plan["march"] == march and plan["generated"] == 1
        if march:
            tx, ty, planes = plan["tile"]
            m = n - 2
            columns = -(-m // tx) * -(-m // ty)
            assert plan["generic_tiles"] == 0 and plan["core_tiles"] % columns == 0
            assert (plan["core_tiles"] // columns) * planes >= m


@pytest.mark.parametrize("make,step,kahan", [
    (lambda: systems.heat1d(101), "resident", False),
    (lambda: systems.brusselator2d(129), "tiles", False),
    (lambda: systems.brusselator2d(801), "sweep", True),
    (lambda: coupled_system(4, 200, True), "tiles", True),
    (lambda: systems.nonlinlap1d(3000, False), "stages", False)])
def test_plan_of_steps(make, step, kahan):
    plan = molgpu.discretize(*make()).plan()
    assert plan["step"] == step and (plan["kahan_waves"] > 0) == kahan and (plan["fused_tiles"] > 0) == (step != "stages")


def test_plan_of_batches(monkeypatch):
    lows = [lower(*systems.diffreact2d(n, 0.05, 1.0, (0, 1, 1, 0))) for n in (20, 90)]
    assert BatchProblem(lows).plan()["step_waves"] > 0
    monkeypatch.setenv("MOL_SWEEP", "0")
    assert BatchProblem(lows).plan()["step_waves"] == 0
