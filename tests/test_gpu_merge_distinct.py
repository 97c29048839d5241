"""The distinct merge of candidates: more images than a launch has waves for, and the edges
of a wave's share of the candidates."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _merge(idx, val, K):
    import torch
    from spinifel_amd import _lib, engine
    engine.require_gpu()
    n, m = idx.shape
    oi = torch.full((n, K), -7, dtype=torch.int32, device="cuda")
    ov = torch.full((n, K), float("nan"), device="cuda")
    P = engine._ptr
    _lib.check(_lib.load().mtip_merge_distinct(P(idx), P(val), n, m, K, P(oi), P(ov), engine._stream()),
               "mtip_merge_distinct")
    return oi, ov


def test_more_images_than_waves():
    """2^26 waves of 64 threads are all that a launch takes."""
    import torch
    n = (1 << 26) + 5
    print(f"case: {n} images", flush=True)
    i = torch.arange(n, dtype=torch.int32, device="cuda")
    idx = torch.stack([i, i ^ 1], 1)
    val = torch.stack([(i % 7).float(), (i % 5).float()], 1)
    oi, ov = _merge(idx, val, 1)
    # the smaller value, of equal ones the smaller index
    first = (val[:, 0] < val[:, 1]) | ((val[:, 0] == val[:, 1]) & (idx[:, 0] < idx[:, 1]))
    assert torch.equal(oi[:, 0], torch.where(first, idx[:, 0], idx[:, 1]))
    assert torch.equal(ov[:, 0], torch.where(first, val[:, 0], val[:, 1]))


@pytest.mark.parametrize("n_in", [1, 63, 64, 65, 130, 512])
@pytest.mark.parametrize("K", [1, 2, 4, 8])
def test_candidates_against_numpy(n_in, K):
    import torch
    rng = np.random.default_rng(n_in + K)
    N = 37
    idx = rng.integers(-1, 40, (N, n_in)).astype(np.int32)
    val = (rng.integers(0, 6, 40)[idx] + 0.5 * (idx % 3)).astype(np.float32)   # by index: repeats are equal
    oi, ov = [t.cpu().numpy() for t in _merge(torch.as_tensor(idx).cuda(), torch.as_tensor(val).cuda(), K)]
    for a, b, x, y in zip(idx, val, oi, ov):
        best = sorted({(float(v), int(k)) for k, v in zip(a, b) if k >= 0})[:K]
        best += [(np.inf, -1)] * (K - len(best))
        assert [(float(v), int(k)) for k, v in zip(x, y)] == best


# the lanes an image has change after 8, 16 and 64 candidates
@pytest.mark.parametrize("n_in", [2, 7, 8, 9, 15, 16, 17, 31, 33])
@pytest.mark.parametrize("K", [1, 2, 4, 8])
@pytest.mark.parametrize("N", [1, 65, 1000])
def test_lanes_an_image(n_in, K, N):
    import torch
    rng = np.random.default_rng(n_in * K + N)
    idx = rng.integers(-1, 12, (N, n_in)).astype(np.int32)
    val = (rng.integers(0, 6, 12)[idx] - 0.5 * (idx % 3)).astype(np.float32)
    oi, ov = [t.cpu().numpy() for t in _merge(torch.as_tensor(idx).cuda(), torch.as_tensor(val).cuda(), K)]
    for a, b, x, y in zip(idx, val, oi, ov):
        best = sorted({(float(v), int(k)) for k, v in zip(a, b) if k >= 0})[:K]
        best += [(np.inf, -1)] * (K - len(best))
        assert [(float(v), int(k)) for k, v in zip(x, y)] == best


def test_more_images_than_waves_of_64_lanes():
    """2^22 workgroups of four images: images past 2^24 are second ones of their waves."""
    import torch
    n, n_in = (1 << 24) + 5, 65
    print(f"case: {n} images of {n_in}", flush=True)
    idx = torch.full((n, n_in), -1, dtype=torch.int32, device="cuda")
    val = torch.zeros((n, n_in), device="cuda")
    i = torch.arange(n, dtype=torch.int32, device="cuda")
    idx[:, 3], val[:, 3] = i, (i % 7).float()
    idx[:, 64], val[:, 64] = i + 1, (i % 5).float()
    oi, ov = _merge(idx, val, 1)
    first = val[:, 3] <= val[:, 64]
    assert torch.equal(oi[:, 0], torch.where(first, i, i + 1))
    assert torch.equal(ov[:, 0], torch.minimum(val[:, 3], val[:, 64]))
