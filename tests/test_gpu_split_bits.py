"""The FP32 cross term gives an image the same bits whatever shares its batch: the kernel
that takes it (by the batch's size), the images beside it, and a NaN or an infinity
among those."""
import numpy as np
import pytest

from helpers import oracle_slicer
from spinifel_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def problem():
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    g = torch.Generator().manual_seed(0)
    S = torch.randn(3092, 80, generator=g).cuda()
    D = torch.randn(3873, 80, generator=g).cuda()
    return S, D, (S.double() ** 2).sum(1)


def _topk(S, D, ss, K=8, tile=128):
    import torch
    from spinifel_amd import engine
    one = torch.ones(1, dtype=torch.float64, device=D.device)
    return engine.topk("fp32", engine.Operand(S, None, ss), ss, len(S), engine.Operand(D.contiguous()),
                       len(D), S.shape[1], one, K, tile=tile)


def _same(a, b):
    import torch
    return torch.equal(a[0], b[0]) and torch.equal(a[1].view(torch.int32), b[1].view(torch.int32))


# 13 x 16 tiles of 256 with a thin last row and column for all images; parts of 1,500 take
# 128-row tiles of four waves (25 x 12 of them), parts of 700 of eight (25 x 6)
@pytest.mark.parametrize("part", [1500, 700, 129, 1])
def test_bits_do_not_depend_on_the_kernel(problem, part):
    S, D, ss = problem
    print(f"case: parts of {part}", flush=True)
    whole = _topk(S, D, ss)
    assert _same(_topk(S, D, ss, tile=256), whole)
    for lo in ([0, 1024, 3173, len(D) - part] if part > 1 else [0, 255, 256, 3840, 3872]):
        rows = slice(lo, min(lo + part, len(D)))
        got = _topk(S, D[rows], ss)
        assert _same(got, (whole[0][rows], whole[1][rows]))


@pytest.mark.parametrize("n", [100, 700, 1500, 3873])
@pytest.mark.parametrize("where", ["image", "slice"])
def test_values_that_are_not_finite_leave_the_others_their_bits(problem, n, where):
    import torch
    S, D, ss = problem
    print(f"case: {n} images, a NaN, an infinity and a huge value in one {where} each", flush=True)
    S, D = S.clone(), D[:n].clone()
    whole = _topk(S, D, ss)
    if where == "image":
        bad = torch.tensor([3, 40, n - 1])
        D[3, 5], D[40, 6], D[n - 1, 7] = float("nan"), float("-inf"), 3.39e38
        got = _topk(S, D, ss)
        keep = torch.ones(n, dtype=torch.bool)
        keep[bad] = False
        keep = keep.cuda()
        assert _same((got[0][keep], got[1][keep]), (whole[0][keep], whole[1][keep]))
        # and those beside none of the three
        assert _same(_topk(S, D[keep], ss), (whole[0][keep], whole[1][keep]))
    else:
        # slices that come last anywhere: all others keep their places and values
        ss = ss.clone()
        bad = torch.tensor([2, 300, 3091])
        ss[bad.cuda()] = 1e30
        S[2, 5], S[300, 6] = float("nan"), float("nan")
        S[3091] *= 2.0 ** 40
        S[3091, 7] = 3.39e38
        D[:, 7].clamp_(min=-1e-30, max=1e-30)
        S2 = S.clone()
        S2[bad.cuda()] = 0
        want, got = [[t.cpu() for t in _topk(s, D, ss)] for s in (S2, S)]
        finite = ~torch.isin(got[0], bad.int())
        assert finite.any(1).all()
        for k in range(n):
            a, b = got[0][k][finite[k]], want[0][k]
            m = len(a)
            assert torch.equal(a, b[:m])
            assert torch.equal(got[1][k][finite[k]].view(torch.int32), want[1][k][:m].view(torch.int32))


def test_fp32_requests_alone_equal_in_mix():
    """Requests of a few images, one of them with a NaN and an infinity, alone and batched."""
    from spinifel_amd import serving
    rng = np.random.default_rng(0)
    srv = serving.Server(precision="fp32", K=4, n_slots=3, max_batch_images=600)
    ac = synth.make_model(33, 120, 1)
    ppr, pdr = synth.detector(1, 32, 32)
    srv.add_model("a", ac, synth.random_quaternions(1200, rng), ppr, pdr)
    sl = oracle_slicer(1e-9)(ac, synth.random_quaternions(300, rng), ppr, pdr.max())
    imgs = synth.poisson_images(sl, 0.5, rng).astype(np.float32)
    reqs = [imgs[rng.choice(300, int(rng.integers(1, 90)), replace=False)].copy() for _ in range(24)]
    reqs[5].reshape(len(reqs[5]), -1)[0, 100] = np.nan
    reqs[11].reshape(len(reqs[11]), -1)[0, 7] = np.inf
    alone = [srv.match_now("a", r) for r in reqs]
    srv.start()
    try:
        mixed = [f.result(timeout=120) for f in [srv.submit("a", r) for r in reqs]]
    finally:
        srv.stop()
    assert max(r.batch_images for r in mixed) > max(len(r) for r in reqs), "no batching happened"
    for k, (a, m) in enumerate(zip(alone, mixed)):
        if k not in (5, 11):
            np.testing.assert_array_equal(a.index, m.index)
            np.testing.assert_array_equal(a.dist64, m.dist64)
