"""The merge operator by pruned DFT matrices, against FFTs in FP64, at the edges of
its tiles and for even, odd and unpadded grids."""
from types import SimpleNamespace

import numpy as np
import pytest

from helpers import rel_l2
from spinifel_amd import synth

pytestmark = pytest.mark.gpu

# five transforms of chains of at most 161 FP64 products, rounding errors adding up
# at most linearly: 5 * 161 * 1.1e-16
TOL = 1e-13

# modes M / 2 + 1 round up to 4, points M_ups / 2 + 1 to 16, columns to 16; more than
# 246 points take more than 64 KiB of LDS
SIZES = [(2, 3), (2, 4), (3, 5), (3, 40), (5, 9), (8, 15), (8, 16), (9, 18), (15, 30), (16, 31),
         (31, 62), (33, 65), (63, 126), (64, 128), (65, 131), (81, 162), (120, 243), (123, 246),
         (124, 248), (130, 260), (160, 320), (20, 320),
         (2, 2), (9, 9), (16, 16), (32, 33), (81, 81), (128, 128), (200, 288), (130, 131), (257, 257),
         (320, 320)]


@pytest.mark.parametrize("M,Mu", SIZES)
def test_convolution_vs_fft(M, Mu):
    import torch
    from spinifel_amd import _lib, engine
    engine.require_gpu()
    print(f"case: M={M} M_ups={Mu}", flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(M * 1000 + Mu)
    K = torch.randn((Mu,) * 3, generator=g, dtype=torch.float64)
    u = torch.randn(M ** 3, generator=g, dtype=torch.float64)
    sup = (torch.rand(M ** 3, generator=g) < 0.7).to(torch.float64)
    F = torch.fft.fftn(torch.fft.rfft(K, dim=0), dim=(1, 2)).contiguous().cuda()
    nbytes = lib.mtip_merge_conv_workspace_size(M, Mu)
    work = torch.full((nbytes // 8,), float("nan"), dtype=torch.float64, device="cuda")
    st, P = engine._stream(), engine._ptr
    _lib.check(lib.mtip_merge_conv_prepare(M, Mu, P(work), nbytes, st), "prepare")
    ud = u.cuda()
    for s in (None, sup):
        v = u if s is None else u * s
        pad = torch.zeros((Mu,) * 3, dtype=torch.float64)
        pad[:M, :M, :M] = v.view(M, M, M)
        y = torch.fft.irfftn(torch.fft.rfftn(pad) * torch.fft.rfftn(K), s=(Mu,) * 3)[:M, :M, :M]
        want = 2.0 * (y.reshape(-1) if s is None else y.reshape(-1) * s) + 0.25 * u
        out = torch.full((M ** 3,), float("nan"), dtype=torch.float64, device="cuda")
        sd = None if s is None else s.cuda()
        for _ in range(2):                     # the workspace is used again
            _lib.check(lib.mtip_merge_conv(P(ud), None if sd is None else P(sd), P(F), M, Mu, 2.0, 0.25,
                                           P(ud), P(work), nbytes, P(out), st), "conv")
        assert rel_l2(out.cpu().numpy(), want.numpy()) <= TOL


def test_refused_sizes():
    from spinifel_amd import _lib
    lib = _lib.load()
    for M, Mu in ((9, 8), (1, 4), (100, 321), (321, 321)):
        assert lib.mtip_merge_conv_workspace_size(M, Mu) == 0
        assert lib.mtip_merge_conv_prepare(M, Mu, 16, 1 << 40, None) == _lib.MTIP_ERR_ARG
    need = lib.mtip_merge_conv_workspace_size(9, 18)
    assert lib.mtip_merge_conv_prepare(9, 18, 16, need - 1, None) == _lib.MTIP_ERR_NOMEM
    assert lib.mtip_merge_conv(16, None, 16, 9, 18, 1.0, 0.0, 16, 16, need - 1, 16,
                               None) == _lib.MTIP_ERR_NOMEM
    assert lib.mtip_merge_conv(16, None, 24, 9, 18, 1.0, 0.0, 16, 16, need, 16,
                               None) == _lib.MTIP_ERR_ARG


@pytest.mark.parametrize("M,Mu", [(21, 30), (21, 42), (20, 40), (20, 45)])
def test_operator_of_a_merge(M, Mu):
    """W against the sum of its terms by FFTs."""
    import torch
    from spinifel_amd.merge import Merge
    ppr, pdr = synth.detector(1, 8, 8)
    s = SimpleNamespace(M=M, M_ups=Mu, oversampling=1.0, solve_ac_maxiter=5)
    mg = Merge(s, np.ones((3, 1, 8, 8), np.float32), ppr, pdr)
    g = torch.Generator().manual_seed(M)
    u = torch.randn(M ** 3, generator=g, dtype=torch.float64).cuda()
    sup = (torch.rand((M,) * 3, generator=g) < 0.7).to(torch.float64).cuda()
    quats = synth.random_quaternions(3, np.random.default_rng(0))
    W, _ = mg.setup_linops(quats, sup, torch.zeros_like(u))
    (x, y, z), _ = mg._points(mg._quats(quats))
    conv = mg._plan_ups.adjoint_points(x, y, z, values=None, out_scale=1.0 / Mu ** 3, spatial=False)
    F = torch.fft.rfftn(torch.fft.ifftshift(conv)) / M ** 3
    want = mg.core_problem_convolution(u, F, sup) + mg.rlambda * u + mg.flambda * mg.fourier_reg(u, sup)
    assert rel_l2(W(u).cpu().numpy(), want.cpu().numpy()) <= TOL
