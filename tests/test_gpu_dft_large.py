"""The fine grid of large models, whose transforms give a wave three output tiles (17 to 24
tiles of 16 points, M from 251), against the closed form of a model of a few voxels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [249, 251, 257, 288, 319, 320])
def test_few_voxels_vs_closed_form(M):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print(f"case: M={M}", flush=True)
    rng = np.random.default_rng(M)
    # the corners and middles of every axis among them
    i = np.concatenate([rng.integers(0, M, (24, 3)), [[0, 0, 0], [M - 1, M - 1, M - 1], [M // 2] * 3,
                                                      [0, M - 1, M // 2], [M // 2 + 1, 0, 1]]])
    i = np.unique(i, axis=0)
    a = rng.uniform(0.5, 2, len(i)).astype(np.float32)
    ac = torch.zeros((M,) * 3, device="cuda")
    ac[tuple(torch.as_tensor(i.T).cuda())] = torch.as_tensor(a).cuda()
    x = rng.uniform(-np.pi, np.pi, (3, 4000))
    x[:, :4] = [[0, np.pi - 1e-9, -np.pi, 1.0]] * 3
    plan = engine.NufftPlan(M, 1e-6, 0)
    plan.set_model(ac)
    got = plan.execute(*[torch.as_tensor(v).cuda() for v in x]).double().cpu().numpy()
    want = (a[:, None].astype(np.float64) * np.cos((i - M // 2) @ x)).sum(0)
    # the kernel's error at eps 1e-6 and its FP32 weights: the bar of the transforms' tests
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
