"""scipy.ndimage.gaussian_filter on device tensors (FP64, separable), for the
three boundary modes the merge and phasing steps use: 'reflect' (the
default, spinifel/sequential/autocorrelation.py:201), 'constant' (cval 0,
spinifel/sequential/phasing.py:258-259) and 'wrap' (:215-216).  The kernel
is scipy's: weights exp(-x^2 / 2 sigma^2) on |x| <= int(truncate sigma + 0.5),
normalised to sum 1, applied along each axis in turn."""
import math

import numpy as np
import torch

from . import _lib, engine

_MODES = {"reflect": 0, "wrap": 1, "constant": 2}
_MAX_RADIUS = 16        # of mtip_gauss_axis


def _index(n, radius, mode, device):
    i = np.arange(-radius, n + radius)
    valid = None
    if mode == "reflect":
        i = np.mod(i, 2 * n)
        i = np.where(i >= n, 2 * n - 1 - i, i)
    elif mode == "wrap":
        i = np.mod(i, n)
    elif mode == "constant":
        valid = (i >= 0) & (i < n)
        i = np.clip(i, 0, n - 1)
    else:
        raise ValueError(f"mode {mode!r}: 'reflect', 'wrap' or 'constant'")
    idx = torch.as_tensor(i, dtype=torch.long, device=device)
    if valid is not None:
        valid = torch.as_tensor(valid, dtype=torch.float64, device=device)
    return idx, valid


def _only_values(t):
    """Whether a tensor is its values and nothing records or transforms what is done
    with it: autograd in either direction, vmap, tracing and subclasses take the
    filter written with torch."""
    return (type(t) in (torch.Tensor, torch.nn.Parameter)
            and not (t.requires_grad and torch.is_grad_enabled())
            and not torch._C._functorch.is_functorch_wrapped_tensor(t)
            and torch.autograd.forward_ad.unpack_dual(t).tangent is None
            and torch.utils._python_dispatch._get_current_dispatch_mode() is None
            and not torch.jit.is_tracing() and not torch.compiler.is_compiling())


def gaussian_filter(a, sigma, mode="reflect", truncate=4.0):
    """gaussian_filter(a, sigma, mode=mode, truncate=truncate) of a device tensor."""
    radius = int(truncate * float(sigma) + 0.5)
    x = np.arange(-radius, radius + 1, dtype=np.float64)
    w = np.exp(-0.5 * (x / sigma) ** 2)
    w /= w.sum()
    out = a.to(torch.float64)
    if out.is_cuda and out.numel() and 0 <= radius <= _MAX_RADIUS and mode in _MODES \
            and out.numel() < 1 << 30 and _only_values(out):
        with torch.cuda.device(out.device):
            r = _filter_axes(out.resolve_neg().contiguous(), w, radius, _MODES[mode])
            # the layout that the loop's zeros_like gives the result of a dense view
            return r if out.is_contiguous() else torch.empty_like(out).copy_(r)
    for ax in range(out.dim()):
        n = out.shape[ax]
        idx, valid = _index(n, radius, mode, out.device)
        pad = out.index_select(ax, idx)
        if valid is not None:
            shape = [1] * out.dim()
            shape[ax] = valid.numel()
            pad = pad * valid.view(shape)
        acc = torch.zeros_like(out)
        for t in range(2 * radius + 1):
            acc += float(w[t]) * pad.narrow(ax, t, n)
        out = acc
    return out


def _filter_axes(a, w, radius, mode):
    """The loop of ``gaussian_filter``, one kernel an axis (the same products and sums in the same
    order, so the same bits)."""
    lib, P, st = _lib.load(), engine._ptr, engine._stream()
    w = np.ascontiguousarray(w, np.float64)
    for ax, n in enumerate(a.shape):
        out = torch.empty_like(a)
        _lib.check(lib.mtip_gauss_axis(P(a), math.prod(a.shape[:ax]), n, math.prod(a.shape[ax + 1:]),
                                       radius, w.ctypes.data, mode, P(out), st), "mtip_gauss_axis")
        a = out
    return a
