"""Grouping of entries by winner at the edges of the scans' shares (1,024 groups a
workgroup, one workgroup alone without a pass for the sums): every entry once, by group."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_groups", [1, 2, 63, 1023, 1024, 1025, 2048, 70001])
@pytest.mark.parametrize("N_i,T", [(1, 1), (700, 3), (5000, 1)])
def test_permutation(n_groups, N_i, T):
    import torch
    from spinifel_amd import _lib, engine
    engine.require_gpu()
    print(f"case: {n_groups} groups, {N_i} x {T} entries", flush=True)
    rng = np.random.default_rng(n_groups + N_i)
    win = rng.integers(-1, n_groups + 1, (N_i, T)).astype(np.int32)     # -1 and n_groups: left out
    lib, P, st = _lib.load(), engine._ptr, engine._stream()
    nb = int(lib.mtip_group_workspace_size(N_i * T, n_groups))
    ws = torch.full((nb,), 0x5a, dtype=torch.uint8, device="cuda")
    w = torch.as_tensor(win).cuda()
    for _ in range(2):
        _lib.check(lib.mtip_group_by_winner(P(w), T, T, N_i, n_groups, P(ws), nb, st), "group")
    po = int(lib.mtip_group_perm_offset(N_i * T, n_groups))
    perm = ws[po:po + 4 * N_i * T].view(torch.int32).cpu().numpy()
    flat = win.reshape(-1)
    assert np.array_equal(np.sort(perm), np.arange(flat.size))
    kept = (flat >= 0) & (flat < n_groups)
    n = int(kept.sum())
    assert kept[perm[:n]].all() and not kept[perm[n:]].any()
    assert (np.diff(flat[perm[:n]]) >= 0).all()
