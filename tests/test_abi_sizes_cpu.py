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
