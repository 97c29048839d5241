"""The pixel-tiling rule by the kernel's width: narrow kernels keep 16 x 16 blocks on
grids of up to 200 points."""
from types import SimpleNamespace

import pytest

from spinifel_amd import engine


@pytest.mark.parametrize("width,det,n,shape", [
    (2, (1, 16, 16), 90, (16, 16)), (4, (1, 32, 32), 90, (16, 16)), (4, (1, 64, 64), 200, (16, 16)),
    (4, (1, 64, 64), 216, (8, 8)), (4, (1, 160, 160), 216, (16, 16)), (5, (1, 32, 32), 90, (16, 16)),
    (5, (1, 32, 32), 100, (16, 16)), (5, (1, 32, 32), 108, (8, 8)), (5, (1, 90, 90), 162, (16, 16)),
    (5, (1, 64, 64), 162, (8, 8)), (5, (1, 108, 108), 216, (8, 8)), (6, (1, 32, 32), 90, (8, 8)),
    (7, (1, 90, 90), 162, (8, 8)), (7, (4, 32, 128), 162, (16, 16))])
def test_rule(width, det, n, shape):
    assert tuple(engine.auto_tiling(SimpleNamespace(n_fine=n, width=width), det).shape) == shape
