"""The transform of the spread grid back to modes by DFT matrices, at the edges of its
tiles, against the direct FP64 sum."""
import numpy as np
import pytest

from helpers import rel_l2
from oracle import es_nufft

pytestmark = pytest.mark.gpu


# n / 2 + 1 points round up to 4, h + 1 modes to 16, columns to 16; 238 takes more than
# 64 KiB of LDS, 256 nine output tiles
@pytest.mark.parametrize("M", [2, 3, 4, 7, 15, 30, 31, 32, 33, 63, 64, 81, 120, 128])
def test_adjoint_of_points_vs_direct_sum(M):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print(f"case: M={M}", flush=True)
    rng = np.random.default_rng(M)
    x = rng.uniform(-np.pi, np.pi, (3, 40))
    x[0, :6] = [-np.pi, np.pi - 1e-9, 0.0, -np.pi, 3.0, -3.1]
    x[2, 2:8] = [-np.pi, np.pi - 1e-9, 0.0, -np.pi, 3.14, -3.14]
    c = rng.standard_normal(40).astype(np.float32)
    plan = engine.NufftPlan(M, 1e-6, 0)
    xs = [torch.as_tensor(v).cuda() for v in x]
    sup = (rng.uniform(size=(M,) * 3) > 0.3).astype(np.float64)
    for s in (None, sup):
        out = plan.adjoint_points(*xs, values=torch.as_tensor(c).cuda(), out_scale=0.5,
                                  support=None if s is None else torch.as_tensor(s).cuda())
        want = 0.5 * es_nufft.nudft3d1(x[0], x[1], x[2], c.astype(np.float64), M, 1).real
        if s is not None:
            want = want * s
        # the kernel's error at eps 1e-6 and its FP32 weights: the adjoint tests' bar
        assert rel_l2(out.cpu().numpy(), want) <= 1e-5


@pytest.mark.parametrize("M", [238, 256, 320])
def test_large_grids_vs_a_plane_wave(M):
    """One point: every mode has the same modulus and a known phase."""
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print(f"case: M={M}", flush=True)
    plan = engine.NufftPlan(M, 1e-6, 0)
    p = (0.7, -2.9, 3.0)
    xs = [torch.tensor([v], dtype=torch.float64).cuda() for v in p]
    out = plan.adjoint_points(*xs, values=torch.ones(1).cuda(), out_scale=1.0).cpu().numpy()
    k = np.arange(M) - M // 2
    e = [np.exp(1j * k * v) for v in p]
    want = (e[0][:, None, None] * (e[1][:, None] * e[2][None, :])[None]).real
    assert rel_l2(out, want) <= 1e-5
