"""The merge rounds as it always has.  Its iteration, stopped far from convergence,
amplifies a rounding of 1e-16 in the kernel, the data term or the operator to 1e-4 and
more of the result, so another order of the sums anywhere would change what solve_ac
returns.  The golden results were written by the revision before the transforms by DFT
matrices came (``python tests/test_gpu_merge_bits.py FILE`` writes them); every
spread of these problems is one run of 128 points whose box fits LDS, so the FP64
atomics add each cell once and the results do not depend on scheduling."""
import os
from types import SimpleNamespace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "merge_bits.npz")
SIZES = [(9, 12), (8, 12), (9, 9), (6, 12)]


def _merge(M, Mu, extent=1.0):
    """Two images of 8 x 8 pixels on a slightly curved surface, nearly the same orientation;
    extent: how far out the points lie, 1 for the grid's edge."""
    from spinifel_amd.merge import Merge
    rng = np.random.default_rng(M)
    g = np.linspace(-1, 1, 8)
    q = np.zeros((3, 1, 8, 8))
    q[0, 0] = g[:, None]
    q[1, 0] = g[None, :]
    q[2, 0] = 0.05 * (g[:, None] ** 2 + g[None] ** 2)
    dist = np.sqrt((q ** 2).sum(0))
    s = SimpleNamespace(M=M, M_ups=Mu, oversampling=1, solve_ac_maxiter=30, nufft_eps=1e-6, device=0)
    quats = np.array([[1.0, 0, 0, 0], [0.999, 0.02, 0.01, 0.03]])
    quats /= np.linalg.norm(quats, axis=1)[:, None]
    return Merge(s, rng.uniform(0.5, 2, (2, 1, 8, 8)).astype(np.float32), extent * q, dist), quats


def _solve(M, Mu):
    mg, quats = _merge(M, Mu)
    return mg.solve_ac(0, quats)


@pytest.mark.parametrize("M,Mu", SIZES)
def test_solve_gives_the_bits_of_the_golden(M, Mu):
    print(f"case: M={M} M_ups={Mu}", flush=True)
    want = np.load(GOLDEN)[f"ac_{M}_{Mu}"]
    for _ in range(2):
        np.testing.assert_array_equal(_solve(M, Mu), want)


@pytest.mark.parametrize("M,Mu", [(20, 40), (21, 45), (33, 66), (81, 162)])
def test_operator_gives_the_bits_of_the_real_transforms(M, Mu):
    """W against the padding, torch's real-to-complex transforms and the recombination."""
    import torch
    from spinifel_amd import _lib, engine
    print(f"case: M={M} M_ups={Mu}", flush=True)
    mg, quats = _merge(M, Mu, extent=0.05)
    g = torch.Generator().manual_seed(M)
    u = torch.randn(M ** 3, generator=g, dtype=torch.float64).cuda()
    sup = (torch.rand((M,) * 3, generator=g) < 0.7).double().cuda()
    W, _ = mg.setup_linops(quats, sup, torch.zeros_like(u))
    (x, y, z), _ = mg._points(mg._quats(quats))
    conv = mg._plan_ups.adjoint_points(x, y, z, values=None, out_scale=1.0 / Mu ** 3, spatial=False,
                                       ordered=True)
    F = torch.fft.rfftn(torch.fft.ifftshift(conv)) / M ** 3
    us = u.view(M, M, M) * sup
    ups = torch.zeros((Mu,) * 3, dtype=torch.float64, device="cuda")
    ups[:M, :M, :M] = us
    X = torch.fft.rfftn(ups)
    X *= F
    y_ups = torch.fft.irfftn(X, s=(Mu,) * 3).contiguous()
    R = torch.fft.rfftn(us)
    R *= mg._reg_mask
    y_reg = torch.fft.irfftn(R, s=(M,) * 3).contiguous()
    want, P = torch.empty_like(u), engine._ptr
    _lib.check(_lib.load().mtip_merge_combine(P(y_ups), P(y_reg), P(u), P(sup), M, Mu, mg.rlambda,
                                              mg.flambda, P(want), engine._stream()), "combine")
    for _ in range(2):
        assert torch.equal(W(u), want)


# complex transforms from 53 on and for factors above 17, real ones otherwise
@pytest.mark.parametrize("M", [3, 17, 19, 37, 49, 51, 53, 55])
def test_regulariser_on_both_sides_of_its_rule(M):
    import torch
    from spinifel_amd import _lib, engine, merge
    engine.require_gpu()
    print(f"case: M={M}", flush=True)
    g = torch.Generator().manual_seed(M)
    u = torch.randn(M ** 3, generator=g, dtype=torch.float64).cuda()
    sup = (torch.rand((M,) * 3, generator=g) < 0.7).double().cuda()
    mask = torch.rand((M, M, M // 2 + 1), generator=g, dtype=torch.float64).cuda()
    us = u.view(M, M, M) * sup
    R = torch.fft.rfftn(us)
    R *= mask
    want = torch.fft.irfftn(R, s=(M,) * 3)
    reg = merge._Regulariser(_lib.load(), M, mask)
    for _ in range(2):
        assert torch.equal(reg.values(u, sup, us), want)


if __name__ == "__main__":
    import sys
    np.savez_compressed(sys.argv[1], **{f"ac_{M}_{Mu}": _solve(M, Mu) for M, Mu in SIZES})
