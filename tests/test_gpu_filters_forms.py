"""The Gaussian filter's kernel against the filter written with torch, in the forms of a call
that the kernel could lose."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def a():
    import torch
    from spinifel_amd import engine
    engine.require_gpu()
    g = torch.Generator(device="cuda").manual_seed(0)
    return torch.randn(6, 8, 10, generator=g, dtype=torch.float64, device="cuda")


def _both(t, *args):
    from spinifel_amd import filters
    return filters.gaussian_filter(t, *args), filters.gaussian_filter(t.cpu(), *args)


@pytest.mark.parametrize("mode", ["reflect", "wrap", "constant"])
@pytest.mark.parametrize("view", ["plain", "permuted", "transposed", "sliced", "expanded", "real"])
def test_result_has_the_layout_of_its_input(a, view, mode):
    import torch
    v = {"plain": lambda: a, "permuted": lambda: a.permute(2, 0, 1), "transposed": lambda: a[0].T,
         "sliced": lambda: a.permute(1, 0, 2)[::2, :, 1::3], "expanded": lambda: a[:, :1].expand(6, 8, 10),
         "real": lambda: torch.complex(a, a).transpose(0, 2).real}[view]()
    got, want = _both(v, 1.0, mode)
    like = torch.zeros_like(v)
    assert got.stride() == like.stride()
    # products and sums of the same values in the same order
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("sigma,truncate", [(-1.0, 4.0), (1.0, -4.0), (-0.1, 4.0), (4.1, 4.0), (4.2, 4.0)])
def test_radii_at_the_ends_of_the_kernels_range(a, sigma, truncate):
    """Below zero the filter is an empty sum; 16 is the kernel's largest, 17 the first beyond."""
    import torch
    got, want = _both(a, sigma, "reflect", truncate)
    assert torch.equal(got.cpu(), want)
