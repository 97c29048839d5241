"""The FP32 cross term with rows of very small values, whose three bf16 parts do not all
exist, against FP64; the rows beside them keep their bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _topk(S, D, K, tile):
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    s, d = torch.as_tensor(S).cuda(), torch.as_tensor(D).cuda()
    ss = torch.zeros(len(S), dtype=torch.float64, device="cuda")
    one = torch.ones(1, dtype=torch.float64, device="cuda")
    idx, val = engine.topk("fp32", engine.Operand(s, None, ss), ss, len(S), engine.Operand(d),
                           len(D), S.shape[1], one, K, tile=tile)
    return idx.cpu().numpy(), val.cpu().numpy()


# around the least exponents at which the parts are exact (2^-110) and the rule's line
# (2^-95), down to denormal values; tiles of 128 in eight and in four waves, of 256 with a
# thin edge
@pytest.mark.parametrize("e", [-90, -95, -97, -108, -112, -116, -122, -126, -135])
@pytest.mark.parametrize("N_o,N_i,tile", [(300, 200, 128), (2100, 2050, 128), (3092, 3873, 128),
                                          (700, 300, 256)])
def test_small_rows_against_fp64(e, N_o, N_i, tile):
    print(f"case: rows of 2^{e}, {N_o} x {N_i}, tile {tile}", flush=True)
    N_p = 112
    rng = np.random.default_rng(-e)
    S = rng.standard_normal((N_o, N_p)).astype(np.float32)
    D = rng.standard_normal((N_i, N_p)).astype(np.float32)
    whole = _topk(S, D, 4, tile)
    # all slices small, images large enough for ordinary products, and the other way round
    for A, B in ((S * 2.0 ** e, D * 2.0 ** 100), (S * 2.0 ** 100, D * 2.0 ** e)):
        A, B = A.astype(np.float32), B.astype(np.float32)
        idx, val = _topk(A, B, 4, tile)
        a, b = A.astype(np.float64), B.astype(np.float64)
        v, mag = -2 * b @ a.T, 2 * np.abs(b) @ np.abs(a).T
        # a rounding a pixel of partial sums below the sum of |a b|, and the value's own
        tol = 2.0 ** -24 * (N_p + 2) * mag
        got = np.take_along_axis(v, idx.astype(np.int64), 1)
        assert (np.abs(val - got) <= np.take_along_axis(tol, idx.astype(np.int64), 1)).all()
        assert (got <= np.sort(v, 1)[:, :4] + 2 * tol.max(1, keepdims=True)).all()
    # a few small images among ordinary ones: those keep their bits
    D2 = D.copy()
    D2[[3, N_i // 2, N_i - 1]] = (D[[3, N_i // 2, N_i - 1]] * 2.0 ** e).astype(np.float32)
    keep = np.setdiff1d(np.arange(N_i), [3, N_i // 2, N_i - 1])
    idx, val = _topk(S, D2, 4, tile)
    np.testing.assert_array_equal(idx[keep], whole[0][keep])
    np.testing.assert_array_equal(val[keep].view(np.int32), whole[1][keep].view(np.int32))
