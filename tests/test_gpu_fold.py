"""Counting sorts around 64 partitions of 1024, up to which a scatter sums the
partitions' counts itself and beyond which a scan kernel does.

The sorted ids and bins must equal the oracle's (tile, depth bits, id) order
exactly: on 16 x 16 tiles (one radix pass of the pairs), on 17 x 17 (row
binning), and with a depth sort of the Gaussians (many pairs each).
"""

import numpy as np
import pytest

import oracle
from tests import helpers as H

pytestmark = pytest.mark.gpu

BW = 16


@pytest.mark.parametrize("n", [65535, 65536, 65537])
@pytest.mark.parametrize("side,radius", [(16, 1), (17, 1), (17, 30)])
def test_partition_edges(n, side, radius):
    rng = np.random.default_rng(n + side)
    tile = rng.integers(0, side * side, n)
    xys = (np.stack([tile % side, tile // side], 1) * BW + BW / 2).astype(np.float32)
    radii = np.full(n, radius, np.int32)
    bits = np.array(2.0, np.float32).view(np.uint32) + rng.integers(0, n // 3, n)
    depths = bits.astype(np.uint32).view(np.float32)
    img = (side * BW, side * BW)
    x0, x1, y0, y1 = oracle.project.tile_rect(xys[:, 0], xys[:, 1], radii.astype(np.float32),
                                              side, side, BW)
    cum = np.cumsum((x1 - x0) * (y1 - y0)).astype(np.int32)
    assert (cum[-1] == n) if radius == 1 else cum[-1] > 16 * n
    gids, _, bins, isect = H.gpu_bin(xys, depths, radii, cum, img_shape=img, block_width=BW,
                                     rects=True)
    _, gs, bs = oracle.binning.bin_and_sort(xys, depths, radii, cum, img_shape=img,
                                            block_width=BW)
    assert isect == cum[-1]
    assert np.array_equal(gids, gs)
    assert np.array_equal(bins, bs)
