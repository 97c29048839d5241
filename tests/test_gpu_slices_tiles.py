"""Slicing with several tiles per 256-point trip: the value of a point does not
depend on the tile it is computed in, so every tiling gives the same bits."""
import numpy as np
import pytest

from spinifel_amd import synth

pytestmark = pytest.mark.gpu


# detectors whose blocks leave a part of the last trip empty, one block, three pixels;
# M = 41 leaves most boxes unstaged at (8, 16), M = 161 some at (8, 8)
@pytest.mark.parametrize("eps", [1e-2, 1e-6, 1e-9])
@pytest.mark.parametrize("M,det", [(41, (1, 32, 32)), (81, (3, 24, 40)), (81, (1, 8, 8)),
                                   (21, (1, 1, 3)), (161, (2, 31, 47))])
def test_same_bits_in_every_tiling(M, det, eps):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print(f"case: M={M} det={det} eps={eps}", flush=True)
    rng = np.random.default_rng(M)
    ac = rng.standard_normal((M, M, M)).astype(np.float32)
    ppr, pdr = synth.detector(*det)
    quats = torch.as_tensor(synth.random_quaternions(5, np.random.default_rng(3)))
    q = torch.as_tensor(np.ascontiguousarray(ppr.reshape(3, -1)))
    n_p = q.shape[1]
    plan = engine.NufftPlan(M, eps, 0)
    plan.set_model(ac)
    scale = np.pi / pdr.max()
    ref = plan.slices(quats, q, scale)
    want = ref["s32"][:, :n_p].cpu().numpy()
    assert np.isfinite(want).all()
    for tile in ((8, 8), (8, 16), (16, 16)):
        r = plan.slices(quats, q, scale, order=engine.tiling(det, tile))
        np.testing.assert_array_equal(r["s32"][:, :n_p].cpu().numpy(), want)
        # FP64 sums of n_p terms in another order
        s = want.astype(np.float64)
        tol = n_p * 2.0 ** -52 * np.abs(s).sum(1)
        assert (np.abs(r["row_sum"].cpu().numpy() - s.sum(1)) <= tol).all()


@pytest.mark.parametrize("tile", [None, (8, 8), (8, 16), (16, 16)])
def test_few_orientations_give_the_bits_of_many(tile):
    """2,048 pixels are one workgroup's work with 1,600 orientations, eight
    workgroups' with seven of them."""
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    print(f"case: tile={tile}", flush=True)
    M, det = 21, (1, 16, 128)
    ac = np.random.default_rng(0).standard_normal((M, M, M)).astype(np.float32)
    ppr, pdr = synth.detector(*det)
    quats = torch.as_tensor(synth.random_quaternions(1600, np.random.default_rng(3)))
    q = torch.as_tensor(np.ascontiguousarray(ppr.reshape(3, -1)))
    plan = engine.NufftPlan(M, 1e-6, 0)
    plan.set_model(ac)
    order = engine.tiling(det, tile) if tile else None
    many = plan.slices(quats, q, np.pi / pdr.max(), order=order)
    few = plan.slices(quats[100:107], q, np.pi / pdr.max(), order=order)
    assert torch.equal(few["s32"], many["s32"][100:107])
    s = few["s32"][:, :2048].double()
    # FP64 sums of 2,048 terms in another order
    for name, terms in (("row_sum", s), ("row_sumsq", s * s)):
        tol = 2048 * 2.0 ** -52 * terms.abs().sum(1)
        assert bool(((few[name] - many[name][100:107]).abs() <= tol).all()), name
        assert bool(((few[name] - terms.sum(1)).abs() <= tol).all()), name
