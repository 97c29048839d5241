"""Sizes that the entry points refuse, or take without overflow, before any GPU work."""
import ctypes

import numpy as np

from spinifel_amd import _lib

FAKE = ctypes.c_void_p(0x1000)      # never dereferenced: the sizes are refused first
OTHER = ctypes.c_void_p(0x2000)


def _gauss(outer, n, inner, radius=1, mode=0):
    w = np.ones(33)
    return _lib.load().mtip_gauss_axis(FAKE, outer, n, inner, radius, w.ctypes.data, mode, OTHER, None)


def test_filter_positions_stay_in_an_int():
    # a position is reflected modulo 2 n
    for n in (1 << 30, (1 << 31) - 1):
        assert _gauss(1, n, 1) == _lib.MTIP_ERR_ARG
        assert "2^30" in _lib.last_error()


def test_filter_counts_do_not_overflow():
    # the product of the three is 2^64 and 2^65 + 2^33: zero and small, modulo 2^64
    for outer, n, inner in ((1 << 32, 1 << 20, 1 << 12), (1 << 33, 1, (1 << 32) + 1)):
        assert _gauss(outer, n, inner) == _lib.MTIP_ERR_ARG
        assert "too many" in _lib.last_error()
    assert _gauss(0, 5, 1 << 40) == _lib.MTIP_OK and _gauss(1 << 40, 5, 0) == _lib.MTIP_OK


def test_regulariser_counts_that_a_launch_does_not_take():
    lib = _lib.load()
    for n in (1 << 32, 1 << 40):
        for rc in (lib.mtip_merge_reg_embed(FAKE, FAKE, n, OTHER, None),
                   lib.mtip_merge_reg_mask(OTHER, FAKE, n, None),
                   lib.mtip_merge_reg_add(FAKE, 1.0, FAKE, 1.0, n, OTHER, None)):
            assert rc == _lib.MTIP_ERR_ARG and "too many" in _lib.last_error()


def test_refusals_of_the_convolution_and_the_half_spectrum():
    """Where a GPU is present a check that went missing would let a kernel run on these
    pointers: here it fails as an error that is not the refusal."""
    lib = _lib.load()
    nul = ctypes.c_void_p()
    for M, Mu in ((9, 8), (1, 4), (100, 321), (321, 321)):
        assert lib.mtip_merge_conv_workspace_size(M, Mu) == 0
        assert lib.mtip_merge_conv_prepare(M, Mu, FAKE, 1 << 40, nul) == _lib.MTIP_ERR_ARG
        assert lib.mtip_merge_conv(FAKE, nul, FAKE, M, Mu, 1.0, 0.0, FAKE, FAKE, 1 << 40, OTHER,
                                   nul) == _lib.MTIP_ERR_ARG
    need = lib.mtip_merge_conv_workspace_size(9, 18)
    assert need > 0 and need % 16 == 0
    odd = ctypes.c_void_p(0x1008)

    def conv(u=FAKE, F=FAKE, base=FAKE, work=FAKE, size=need, out=OTHER):
        return lib.mtip_merge_conv(u, nul, F, 9, 18, 1.0, 0.0, base, work, size, out, nul)

    assert lib.mtip_merge_conv_prepare(9, 18, FAKE, need - 1, nul) == _lib.MTIP_ERR_NOMEM
    assert lib.mtip_merge_conv_prepare(9, 18, nul, need, nul) == _lib.MTIP_ERR_ARG
    assert conv(size=need - 1) == _lib.MTIP_ERR_NOMEM
    for bad in (dict(F=odd), dict(work=odd), dict(u=nul), dict(F=nul), dict(base=nul), dict(work=nul),
                dict(out=nul)):
        assert conv(**bad) == _lib.MTIP_ERR_ARG, bad
    for M in (-1, 0, 2, 80, 2049):
        assert lib.mtip_half_pack(FAKE, M, OTHER, nul) == _lib.MTIP_ERR_ARG
        assert lib.mtip_half_expand(FAKE, M, OTHER, nul) == _lib.MTIP_ERR_ARG
    assert lib.mtip_half_pack(nul, 9, OTHER, nul) == _lib.MTIP_ERR_ARG
    assert lib.mtip_half_expand(FAKE, 9, nul, nul) == _lib.MTIP_ERR_ARG
    assert lib.mtip_merge_reg_embed(FAKE, nul, 4, OTHER, nul) == _lib.MTIP_ERR_ARG
    assert lib.mtip_merge_reg_mask(OTHER, FAKE, 0, nul) == _lib.MTIP_ERR_ARG
    assert lib.mtip_merge_reg_add(nul, 1.0, FAKE, 1.0, 4, OTHER, nul) == _lib.MTIP_ERR_ARG
    assert lib.mtip_plan_spread_finish_ordered(nul, nul, 1.0, OTHER, nul) == _lib.MTIP_ERR_ARG
