"""Slices of few and many orientations by kernels of several widths, where the split of an
orientation among workgroups begins: one set of values, and FP64 sums of them."""
import numpy as np
import pytest

from spinifel_amd import synth

pytestmark = pytest.mark.gpu


# an orientation is split from 14 trips of 256 points times the kernel's width on, 256-point
# tiles not from 2,048 (up to 4 points wide) or 4,096 orientations on
@pytest.mark.parametrize("eps", [1e-1, 1e-3, 1e-4, 1e-6])
@pytest.mark.parametrize("trips", [2, 3, 4, 7])
@pytest.mark.parametrize("tile", [None, (8, 8)])
def test_values_and_sums(eps, trips, tile):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print(f"case: eps={eps} trips={trips} tile={tile}", flush=True)
    M, det = 15, (1, 16, 16 * trips - 3)
    ac = np.random.default_rng(trips).standard_normal((M, M, M)).astype(np.float32)
    ppr, pdr = synth.detector(*det)
    quats = torch.as_tensor(synth.random_quaternions(4100, np.random.default_rng(3)))
    q = torch.as_tensor(np.ascontiguousarray(ppr.reshape(3, -1)))
    n_p = q.shape[1]
    plan = engine.NufftPlan(M, eps, 0)
    plan.set_model(ac)
    order = engine.tiling(det, tile) if tile else None
    many = plan.slices(quats, q, np.pi / pdr.max(), order=order)
    for n in (1, 100, 2047, 2048):
        few = plan.slices(quats[:n], q, np.pi / pdr.max(), order=order)
        assert torch.equal(few["s32"], many["s32"][:n])
        s = few["s32"][:, :n_p].double()
        assert bool(torch.isfinite(s).all())
        for name, terms in (("row_sum", s), ("row_sumsq", s * s)):
            # FP64 sums of n_p terms in another order
            tol = n_p * 2.0 ** -52 * terms.abs().sum(1)
            assert bool(((few[name] - terms.sum(1)).abs() <= tol).all()), name
            assert bool(((many[name][:n] - terms.sum(1)).abs() <= tol).all()), name
