"""The half-spectrum layout kernels and the regulariser on them (odd edges), against
torch's real-to-complex transforms, bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


# 64 rows (M^2) x 16 columns (M / 2 + 1) a tile
@pytest.mark.parametrize("M", [1, 3, 5, 9, 29, 31, 33, 63, 81, 101])
def test_half_spectrum_layouts(M):
    import torch
    from spinifel_amd import _lib, engine
    engine.require_gpu()
    print(f"case: M={M}", flush=True)
    lib, P, st = _lib.load(), engine._ptr, engine._stream()
    g = torch.Generator(device="cuda").manual_seed(M)
    F = torch.randn(M, M, M, generator=g, dtype=torch.complex128, device="cuda")
    h = M // 2 + 1
    Y = torch.full((h, M, M), float("nan"), dtype=torch.complex128, device="cuda")
    _lib.check(lib.mtip_half_pack(P(F), M, P(Y), st), "pack")
    assert torch.equal(Y, F[..., :h].permute(2, 0, 1))
    W = torch.full((M, M, M), float("nan"), dtype=torch.complex128, device="cuda")
    _lib.check(lib.mtip_half_expand(P(Y), M, P(W), st), "expand")
    want = torch.cat([F[..., :h], F[..., 1:h].flip(-1).conj()], dim=2)
    assert torch.equal(W, want)


@pytest.mark.parametrize("M", [9, 20, 33, 57, 81])
def test_regulariser_gives_the_bits_of_the_real_transforms(M):
    import torch
    from spinifel_amd import _lib, engine, merge
    engine.require_gpu()
    print(f"case: M={M}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M)
    u = torch.randn(M ** 3, generator=g, dtype=torch.float64, device="cuda")
    sup = (torch.rand(M, M, M, generator=g, device="cuda") < 0.7).double()
    mask = torch.rand(M, M, M // 2 + 1, generator=g, dtype=torch.float64, device="cuda")
    X = torch.fft.rfftn(u.view(M, M, M) * sup)
    X *= mask
    want = (torch.fft.irfftn(X, s=(M,) * 3) * sup).reshape(-1)
    reg = merge._Regulariser(_lib.load(), M, mask)
    for _ in range(2):
        # flambda 1 on zero: nothing but the term itself
        out = torch.zeros_like(u)
        reg(u, sup, 1.0, out)
        assert torch.equal(out, want)


def test_refused_arguments():
    from spinifel_amd import _lib
    lib = _lib.load()
    for M in (0, 2, 80, 2049):
        assert lib.mtip_half_pack(16, M, 16, None) == _lib.MTIP_ERR_ARG
        assert lib.mtip_half_expand(16, M, 16, None) == _lib.MTIP_ERR_ARG
    assert lib.mtip_half_pack(None, 9, 16, None) == _lib.MTIP_ERR_ARG
    assert lib.mtip_merge_reg_embed(16, None, 4, 16, None) == _lib.MTIP_ERR_ARG
    assert lib.mtip_merge_reg_mask(16, 16, 0, None) == _lib.MTIP_ERR_ARG
    assert lib.mtip_merge_reg_add(None, 1.0, 16, 1.0, 4, 16, None) == _lib.MTIP_ERR_ARG
