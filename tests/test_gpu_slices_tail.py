"""Slices whose last trip of 256 slots has one to three tiles, or a tile without pixels
between others: the values of a plain list of the same pixels, bit for bit."""
import numpy as np
import pytest

from spinifel_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eps", [1e-1, 1e-6, 1e-9, 1e-12])
@pytest.mark.parametrize("det", [(1, 8, 8), (1, 8, 15), (1, 20, 7), (1, 24, 20), (3, 5, 17)])
def test_last_trip(det, eps):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print(f"case: det={det} eps={eps}", flush=True)
    M = 17
    ac = np.random.default_rng(M).standard_normal((M, M, M)).astype(np.float32)
    ppr, pdr = synth.detector(*det)
    quats = torch.as_tensor(synth.random_quaternions(70, np.random.default_rng(3)))
    q = torch.as_tensor(np.ascontiguousarray(ppr.reshape(3, -1)))
    n_p = q.shape[1]
    plan = engine.NufftPlan(M, eps, 0)
    plan.set_model(ac)
    scale = np.pi / pdr.max()
    want = plan.slices(quats, q, scale)["s32"][:, :n_p]
    assert bool(torch.isfinite(want).all())
    for tile in ((8, 8), (8, 16)):
        t = engine.tiling(det, tile)
        order = np.asarray(t.order)
        none = np.full(t.points, -1, np.int32)
        gaps = np.concatenate([none] + [np.concatenate([r, none]) for r in order.reshape(-1, t.points)])
        for o in (order, gaps):
            got = plan.slices(quats, q, scale, order=engine.Tiling(o, t.points, t.shape))
            assert torch.equal(got["s32"][:, :n_p], want)
            # FP64 sums of n_p terms in another order
            s = want.double()
            assert bool(((got["row_sum"] - s.sum(1)).abs() <= n_p * 2.0 ** -52 * s.abs().sum(1)).all())
            assert int(got["bad"].item()) == 0
