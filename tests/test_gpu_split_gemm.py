"""The FP32 cross term (three bf16 parts per value, six partial products)
against FP64, at the edges of its tiles and with values that are not finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    return torch.device("cuda", 0)


def _topk(S, D, K, tile, dev):
    import torch
    from spinifel_amd import engine
    s, d = torch.as_tensor(S).to(dev), torch.as_tensor(D).to(dev)
    ss = (s.double() ** 2).sum(1)
    one = torch.ones(1, dtype=torch.float64, device=dev)
    idx, val = engine.topk("fp32", engine.Operand(s, None, ss), ss, len(S), engine.Operand(d),
                           len(D), S.shape[1], one, K, tile=tile)
    return idx.cpu().numpy(), val.double().cpu().numpy()


# 128-row tiles of eight waves, of four (289 tiles); 13 x 16 tiles of 256 with a thin last row and column (its keys in
# 128-row tiles, an odd number of them) and without; one pixel stage, odd stages
@pytest.mark.parametrize("N_o,N_i,N_p,K", [(1, 1, 80, 1), (127, 129, 112, 8), (129, 300, 208, 4),
                                           (200, 300, 64, 4), (2100, 2050, 96, 8),
                                           (3092, 3873, 80, 4), (3201, 3850, 96, 2),
                                           (3328, 4096, 112, 1)])
@pytest.mark.parametrize("tile", [128, 256])
def test_split_topk_against_fp64(dev, N_o, N_i, N_p, K, tile):
    print(f"case: split FP32 top-{K} {(N_o, N_i, N_p)} tile {tile}", flush=True)
    rng = np.random.default_rng(N_o + N_p)
    # magnitudes over 2^-20 .. 2^20, so that all three parts matter
    S = (rng.standard_normal((N_o, N_p)) * 2.0 ** rng.integers(-20, 20, (1, N_p))).astype(np.float32)
    D = (rng.standard_normal((N_i, N_p)) * 2.0 ** rng.integers(-20, 20, (1, N_p))).astype(np.float32)
    idx, val = _topk(S, D, K, tile, dev)
    s, d = S.astype(np.float64), D.astype(np.float64)
    ss = (s * s).sum(1)
    v = ss[None] - 2 * d @ s.T
    # products dropped and rounded: below 2^-24 |a b| each; 6 roundings per 16
    # pixels of partial sums below sum |a b|, each one unit in the last place;
    # then the value's own rounding
    mag = np.abs(d) @ np.abs(s).T
    tol = 2.0 ** -23 * (2 * mag * (6 * (N_p // 16) + 2) + ss[None] + np.abs(v))
    k = min(K, N_o)
    assert (idx[:, k:] == -1).all()
    got = np.take_along_axis(v, idx[:, :k].astype(np.int64), 1)
    t = np.take_along_axis(tol, idx[:, :k].astype(np.int64), 1)
    assert (np.abs(val[:, :k] - got) <= t).all()
    assert all(len(set(r)) == k for r in idx[:, :k])
    best = np.sort(v, 1)[:, :k]
    assert (got <= best + 2 * tol.max(1, keepdims=True)).all()


@pytest.mark.parametrize("shape", [(300, 200, 96), (3100, 3900, 80)])
def test_split_topk_keeps_infinities(dev, shape):
    N_o, N_i, N_p = shape
    print(f"case: split FP32 top-K with infinities {shape}", flush=True)
    rng = np.random.default_rng(4)
    S = rng.standard_normal((N_o, N_p)).astype(np.float32)
    D = rng.standard_normal((N_i, N_p)).astype(np.float32)
    S[5, 7] = np.inf
    D[:, 7][D[:, 7] == 0] = 1.0
    S[200, 3] = 3.39e38        # rounds to an infinite bf16
    D[11, 3], D[12, 3] = 0.0, 1e-30
    import torch
    from spinifel_amd import engine
    s, d = torch.as_tensor(S).to(dev), torch.as_tensor(D).to(dev)
    ss = torch.full((N_o,), 10.0, dtype=torch.float64, device=dev)
    one = torch.ones(1, dtype=torch.float64, device=dev)
    idx, val = engine.topk("fp32", engine.Operand(s, None, ss), ss, N_o, engine.Operand(d), N_i,
                           N_p, one, 2)
    idx, val = idx.cpu().numpy(), val.cpu().numpy()
    pos = D[:, 7] > 0
    assert (idx[pos, 0] == 5).all() and np.isneginf(val[pos, 0]).all()
    assert (idx[~pos] != 5).all()
    # the large finite slice: its dot with image 11 is an ordinary number
    x = 10.0 - 2.0 * D.astype(np.float64) @ np.where(np.isinf(S), 0, S).astype(np.float64).T
    lo = [i for i in (11, 12) if not pos[i]]
    for i in lo:
        want = np.argsort(x[i] + np.where(np.arange(N_o) == 5, np.inf, 0))[:2]
        np.testing.assert_array_equal(idx[i], want)
