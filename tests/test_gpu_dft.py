"""The pruned transforms by DFT matrices (fine grid of a model) at the edges of
their tiles, against the direct FP64 sum."""
import numpy as np
import pytest

from helpers import nudft_real, rel_l2

pytestmark = pytest.mark.gpu


def _plan(M, eps=1e-6):
    from spinifel_amd import engine
    engine.require_gpu()
    return engine.NufftPlan(M, eps, 0)


# h + 1 modes round up to 4, n / 2 + 1 outputs to 16, columns to 32 (16 above 124 modes)
@pytest.mark.parametrize("M", [2, 3, 4, 7, 15, 30, 31, 32, 33, 62, 63, 64, 124, 125, 246, 248])
def test_grid_of_a_model_vs_direct_sum(M):
    print(f"case: M={M}", flush=True)
    rng = np.random.default_rng(M)
    ac = rng.standard_normal((M, M, M)).astype(np.float32)
    plan = _plan(M)
    plan.set_model(np.zeros_like(ac))
    plan.set_model(ac)                      # a second model leaves nothing of the first
    # points over the whole cell, its edges included (padded copies of the grid)
    x = rng.uniform(-np.pi, np.pi, (3, 30))
    x[0, :6] = [-np.pi, np.pi - 1e-9, 0.0, -np.pi, 3.0, -3.1]
    x[2, 2:8] = [-np.pi, np.pi - 1e-9, 0.0, -np.pi, 3.14, -3.14]
    out = plan.execute(x[0], x[1], x[2]).double().cpu().numpy()
    # kernel error 1e-6 of the sum's norm per point, the FP32 floor of the kernel
    # beside it: the bar of the other transform tests
    err = rel_l2(out, nudft_real(ac, x[0], x[1], x[2]))
    print("rel_l2", err)
    assert err <= 1e-5


def test_non_finite_model_values_reach_every_point():
    M = 21
    ac = np.ones((M, M, M), np.float32)
    ac[3, 4, 5] = np.nan
    plan = _plan(M)
    plan.set_model(ac)
    x = np.random.default_rng(0).uniform(-np.pi, np.pi, (3, 50))
    assert np.isnan(plan.execute(x[0], x[1], x[2]).cpu().numpy()).all()
