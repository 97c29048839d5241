"""The pixel-tiling rule: every pixel once for any detector, block size by the pixel
spacing on the fine grid alone."""
from types import SimpleNamespace

import numpy as np
import pytest

from spinifel_amd import engine


@pytest.mark.parametrize("det,n,shape", [
    ((1, 32, 32), 90, (8, 8)), ((1, 64, 64), 90, (16, 16)), ((4, 32, 128), 162, (16, 16)),
    ((4, 32, 128), 216, (8, 8)), ((3, 37, 128), 250, (8, 8)), ((4, 64, 256), 324, (16, 16)),
    ((1, 1, 7), 18, (8, 8)), ((2, 5, 3), 8, (16, 16)), ((24, 40), 64, (8, 8))])
def test_rule(det, n, shape):
    t = engine.auto_tiling(SimpleNamespace(n_fine=n), det)
    assert tuple(t.shape) == shape and t.points == shape[0] * shape[1]
    order = np.asarray(t.order)
    assert order.size % t.points == 0
    assert np.array_equal(np.sort(order[order >= 0]), np.arange(np.prod(det)))


def test_flat_pixel_lists_have_no_tiling():
    assert engine.auto_tiling(SimpleNamespace(n_fine=90), (1000,)) is None
