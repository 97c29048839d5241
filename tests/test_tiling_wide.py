"""The pixel-tiling rule for kernels of 13 points and more, and for detectors of one block."""
from types import SimpleNamespace

import pytest

from spinifel_amd import engine


@pytest.mark.parametrize("width,det,n,shape", [
    # wide kernels: 16 x 16 up to 200 points, but where padding doubles the slots
    (13, (1, 90, 90), 162, (16, 16)), (15, (1, 48, 50), 90, (16, 16)), (13, (1, 12, 9), 30, (16, 16)),
    (14, (1, 90, 90), 200, (16, 16)), (14, (1, 90, 90), 216, (8, 8)), (14, (1, 24, 20), 90, (8, 8)),
    (13, (1, 8, 8), 50, (8, 8)), (12, (1, 90, 90), 162, (8, 8)),
    # one 16 x 16 block, one 8 x 8 block, two 16 x 16 blocks
    (7, (1, 16, 16), 50, (16, 16)), (6, (12, 9), 200, (16, 16)), (7, (1, 16, 16), 216, (8, 8)),
    (7, (1, 8, 8), 50, (8, 8)), (7, (2, 16, 16), 50, (8, 8)), (8, (1, 16, 16), 50, (8, 8))])
def test_rule(width, det, n, shape):
    assert tuple(engine.auto_tiling(SimpleNamespace(n_fine=n, width=width), det).shape) == shape
