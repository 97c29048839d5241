"""Spreading with the zero values taken out of each tile: all zero, one value a tile,
a tenth, all; tiles of every size, windows of several widths; and the box left clean
between tiles."""
import numpy as np
import pytest

from helpers import normalized_points, rel_l2
from oracle import es_nufft
from spinifel_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eps", [1e-2, 1e-6, 1e-9])
@pytest.mark.parametrize("tile", [None, (8, 8), (8, 16), (16, 16)])
def test_sparse_values_vs_direct_sum(tile, eps):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    M, det, N_o = 16, (3, 20, 40), 3
    ppr, pdr = synth.detector(*det)
    n_p = ppr[0].size
    quats = synth.random_quaternions(N_o, np.random.default_rng(2))
    H, K, L = normalized_points(quats, ppr, pdr.max())
    plan = engine.NufftPlan(M, eps, 0)
    order = engine.tiling(det, tile) if tile else None
    q = torch.as_tensor(np.ascontiguousarray(ppr.reshape(3, -1)))
    rng = np.random.default_rng(5)
    for share in (0.0, 0.01, 0.1, 1.0):
        print(f"case: tile={tile} eps={eps} share={share}", flush=True)
        v = (rng.standard_normal((N_o, n_p)) * (rng.uniform(size=(N_o, n_p)) < share)).astype(np.float32)
        out = plan.adjoint_slices(torch.as_tensor(quats), q, np.pi / pdr.max(), out_scale=1.0,
                                  values=torch.as_tensor(v).cuda(), order=order).cpu().numpy()
        if share == 0.0:
            assert not out.any()
            continue
        want = es_nufft.nudft3d1(H.ravel(), K.ravel(), L.ravel(), v.ravel().astype(np.float64), M, 1).real
        # the kernel's error (a few eps) over its FP32 weights' floor
        assert rel_l2(out, want) <= max(10 * eps, 1e-5)


def test_tiles_beyond_the_box_between_tiles_within():
    """Runs of 256 pixels in index order, alternately one point's window and windows
    across the whole grid (no box): what a tile leaves must not reach the next."""
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print("case: alternating boxes", flush=True)
    M = 61
    rng = np.random.default_rng(1)
    q = rng.uniform(-1, 1, (3, 2048))
    q[:, (np.arange(2048) // 256) % 2 == 0] *= 0.02
    v = rng.standard_normal((1, 2048)).astype(np.float32)
    plan = engine.NufftPlan(M, 1e-6, 0)
    one = torch.tensor([[1.0, 0.0, 0.0, 0.0]], dtype=torch.float64)
    for tiling in (None, engine.Tiling(torch.arange(2048, dtype=torch.int32), 64, (8, 8))):
        out = plan.adjoint_slices(one, torch.as_tensor(q), np.pi, values=torch.as_tensor(v).cuda(),
                                  order=tiling, out_scale=1.0).cpu().numpy()
        x = q * np.pi
        want = es_nufft.nudft3d1(x[0], x[1], x[2], v.ravel().astype(np.float64), M, 1).real
        assert rel_l2(out, want) <= 1e-5
