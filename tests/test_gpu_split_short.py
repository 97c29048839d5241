"""The FP32 cross term around the row lengths at which its kernels change (48 and 128
values for each of the K best): an image's keys have the same bits in a large batch and
in parts of it, and agree with FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _topk(S, D, ss, K, tile=128):
    import torch
    from spinifel_amd import engine
    one = torch.ones(1, dtype=torch.float64, device="cuda")
    return engine.topk("fp32", engine.Operand(S, None, ss), ss, len(S), engine.Operand(D.contiguous()),
                       len(D), S.shape[1], one, K, tile=tile)


# 25 x 31 tiles of 128 with thin edges, 13 x 16 of 256; parts of 1,500 are 25 x 12 tiles,
# parts of 700 25 x 6
@pytest.mark.parametrize("K", [1, 2, 4, 8])
@pytest.mark.parametrize("values", [48, 128])
@pytest.mark.parametrize("past", [False, True])
def test_both_sides_of_the_lines(K, values, past):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    n_pix = max(80, values * K // 16 * 16) + (16 if past else 0)
    print(f"case: {n_pix} values, K={K}", flush=True)
    g = torch.Generator().manual_seed(n_pix + K)
    S = torch.randn(3092, n_pix, generator=g).cuda()
    D = torch.randn(3873, n_pix, generator=g).cuda()
    ss = (S.double() ** 2).sum(1)
    idx, val = _topk(S, D, ss, K)
    for part in (1500, 700):
        rows = slice(3873 - part, 3873)
        i, v = _topk(S, D[rows], ss, K)
        assert torch.equal(i, idx[rows]) and torch.equal(v.view(torch.int32), val[rows].view(torch.int32))
    i, v = _topk(S, D, ss, K, tile=256)
    assert torch.equal(i, idx) and torch.equal(v.view(torch.int32), val.view(torch.int32))
    # a rounding a value of partial sums below the sum of |s d|, and the key's own
    s, d = S.double(), D.double()
    exact = ss[None] - 2 * d @ s.T
    tol = 2.0 ** -24 * (n_pix + 2) * (2 * d.abs() @ s.abs().T) + 2.0 ** -23 * ss[None]
    at = idx.long()
    assert bool(((val.double() - exact.gather(1, at)).abs() <= tol.gather(1, at)).all())
    best = exact.sort(1).values[:, :K]
    assert bool((exact.gather(1, at) <= best + 2 * tol.max(1, keepdim=True).values).all())
