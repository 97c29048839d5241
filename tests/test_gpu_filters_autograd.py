"""The Gaussian filter of device tensors that are more than their values: the filter
written with torch takes them, with and beside the kernel the same values."""
import pytest

pytestmark = pytest.mark.gpu

SIGMA = 1.0


@pytest.fixture(scope="module")
def a():
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    g = torch.Generator(device="cuda").manual_seed(0)
    return torch.randn(5, 6, 7, generator=g, dtype=torch.float64, device="cuda")


def _filter(t, mode="reflect"):
    from spinifel_amd import filters
    return filters.gaussian_filter(t, SIGMA, mode)


@pytest.mark.parametrize("mode", ["reflect", "wrap", "constant"])
def test_backward(a, mode):
    import torch
    x = a.clone().requires_grad_()
    y = _filter(x, mode)
    assert y.requires_grad and torch.equal(y.detach(), _filter(a, mode))
    v = torch.linspace(-1, 1, a.numel(), dtype=torch.float64, device="cuda").view_as(a)
    g, = torch.autograd.grad(y, x, v)
    # <v, F a> = <F^T v, a>: 3 x 9 products and sums of values of order one a voxel
    assert abs(float((v * y.detach()).sum() - (g * a).sum())) <= 1e-12 * a.numel()
    with torch.no_grad():
        assert not _filter(x, mode).requires_grad
        assert torch.equal(_filter(torch.nn.Parameter(a), mode), y)


def test_forward_mode_and_vmap(a):
    import torch
    import torch.autograd.forward_ad as fwd
    t = a.flip(0)
    with fwd.dual_level():
        p, d = fwd.unpack_dual(_filter(fwd.make_dual(a, t)))
        assert torch.equal(p, _filter(a)) and torch.equal(d, _filter(t))
    p, d = torch.func.jvp(_filter, (a,), (t,))
    assert torch.equal(p, _filter(a)) and torch.equal(d, _filter(t))
    # a batch: every slice a filtered 2D array
    got = torch.func.vmap(_filter)(a)
    assert torch.equal(got, torch.stack([_filter(s) for s in a]))


def test_views_with_a_pending_negation(a):
    import torch
    z = torch.complex(a[0], a[1])
    v = z.conj().imag
    assert v.is_neg()
    assert torch.equal(_filter(v), _filter(v.resolve_neg().clone()))
    w = torch._neg_view(a)
    assert w.is_neg() and w.is_contiguous()
    assert torch.equal(_filter(w), _filter(-a))


def test_tracing_records_the_operations(a):
    from torch.fx.experimental.proxy_tensor import make_fx
    import torch
    g = make_fx(lambda t: _filter(t))(a)
    b = a.flip(1).contiguous()
    assert torch.equal(g(b), _filter(b))
