"""The Gaussian filter's kernel against the filter written with torch, bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["reflect", "wrap", "constant"])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 1), (7, 9, 11), (33, 33, 33), (5, 64), (100,)])
def test_filter_gives_the_bits_of_the_loop(shape, mode, monkeypatch):
    import torch
    from spinifel_amd import engine, filters
    engine.require_gpu()
    g = torch.Generator(device="cuda").manual_seed(len(shape))
    a = torch.randn(shape, generator=g, dtype=torch.float64, device="cuda")
    views = [a, a.float(), a.transpose(0, -1)]
    b = a.clone()
    b.view(-1)[0] = float("nan")
    b.view(-1)[-1] = float("inf")
    views.append(b)
    # radius 0, 2, 8, 16 (the kernel's largest; most reach past the array) and 20 (torch)
    for sigma, truncate in ((0.1, 2), (1, 2), (2.0, 4.0), (4.0, 4.0), (5.0, 4.0)):
        for v in views:
            got = filters.gaussian_filter(v, sigma, mode, truncate)
            with monkeypatch.context() as m:
                m.setattr(filters, "_MAX_RADIUS", -1)
                want = filters.gaussian_filter(v, sigma, mode, truncate)
            assert got.shape == want.shape
            assert torch.equal(torch.isnan(got), torch.isnan(want))
            assert torch.equal(got.nan_to_num(0.5), want.nan_to_num(0.5))


def test_unknown_mode_is_refused():
    import torch
    from spinifel_amd import engine, filters
    engine.require_gpu()
    with pytest.raises(ValueError):
        filters.gaussian_filter(torch.zeros(4, 4, device="cuda"), 1, "mirror")
