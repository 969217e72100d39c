"""Binning by tile rows (``csrc/rowbin.hip``) at the edges of its ranges.

The sorted ids, tile ids and bins must equal the oracle's stable (tile, depth
bits, id) order exactly (``oracle.binning``, reference ``lib/ops.cu:722-760``):
one Gaussian more and fewer than a partition (1024), tile grids just inside and
outside the LDS widths (128 and 256 tiles per axis; 257 takes the pair sort),
few pairs per Gaussian (id order, tiles ordered afterwards) and many (depth
order, stable placement), rectangles over the whole grid (more pairs per
partition than the LDS stage holds) and depth ties broken by id.
"""

import numpy as np
import pytest

import oracle
from tests import helpers as H

pytestmark = pytest.mark.gpu

BW = 16


def _scene(n, tiles, radius, seed):
    rng = np.random.default_rng(seed)
    h, w = tiles[0] * BW - 3, tiles[1] * BW - 5          # ragged last row and column
    xys = np.stack([rng.uniform(-10, w + 10, n), rng.uniform(-10, h + 10, n)], 1).astype(np.float32)
    radii = rng.integers(1, radius + 1, n).astype(np.int32)
    radii[rng.random(n) < 0.1] = 0
    radii[: n // 200] = max(h, w) + 20                    # the whole grid
    bits = np.array(2.0, np.float32).view(np.uint32) + rng.integers(0, max(n // 4, 1), n)
    depths = bits.astype(np.uint32).view(np.float32)
    ty, tx = tiles
    x0, x1, y0, y1 = oracle.project.tile_rect(xys[:, 0], xys[:, 1], radii.astype(np.float32), tx,
                                              ty, BW)
    cnt = np.where(radii > 0, (x1 - x0) * (y1 - y0), 0)
    return xys, depths, radii, np.cumsum(cnt).astype(np.int32), (h, w)


@pytest.mark.parametrize("path", [{}, {"rects": True}], ids=["one", "rects"])
@pytest.mark.parametrize("radius", [12, 90], ids=["small", "large"])
@pytest.mark.parametrize("n", [1, 1023, 1025, 6000])
@pytest.mark.parametrize("tiles", [(17, 17), (128, 3), (129, 3), (3, 128), (3, 129), (2, 256),
                                   (2, 257), (256, 2)], ids=str)
def test_row_binning_bitexact(tiles, n, radius, path):
    xys, depths, radii, cum, img = _scene(n, tiles, radius, seed=n + radius + tiles[0])
    gids, tids, bins, isect = H.gpu_bin(xys, depths, radii, cum, img_shape=img, block_width=BW,
                                        **path)
    ks, gs, bs = oracle.binning.bin_and_sort(xys, depths, radii, cum, img_shape=img,
                                             block_width=BW)
    assert isect == ks.size
    assert np.array_equal(gids, gs)
    if isect:
        keys = (tids.astype(np.int64) << 32) | depths.view(np.int32)[gids].astype(np.int64)
        assert np.array_equal(keys, ks)
    assert np.array_equal(bins, bs)


@pytest.mark.parametrize("path", [{}, {"rects": True}], ids=["one", "rects"])
@pytest.mark.parametrize("tiles", [(17, 17), (128, 3), (129, 3), (3, 128), (3, 129), (2, 256),
                                   (256, 2)], ids=str)
def test_depth_order_bitexact(tiles, path):
    """Many pairs per Gaussian and per tile: most rectangles cover the grid."""
    n = 1700
    xys, depths, radii, _, img = _scene(n, tiles, 90, seed=sum(tiles))
    radii[: 6 * n // 10] = max(img) + 20
    perm = np.random.default_rng(5).permutation(n)
    xys, radii = xys[perm], radii[perm]
    x0, x1, y0, y1 = oracle.project.tile_rect(xys[:, 0], xys[:, 1], radii.astype(np.float32),
                                              tiles[1], tiles[0], BW)
    cum = np.cumsum(np.where(radii > 0, (x1 - x0) * (y1 - y0), 0)).astype(np.int32)
    assert cum[-1] > 16 * n and cum[-1] > 640 * tiles[0] * tiles[1]
    gids, tids, bins, isect = H.gpu_bin(xys, depths, radii, cum, img_shape=img, block_width=BW,
                                        **path)
    ks, gs, bs = oracle.binning.bin_and_sort(xys, depths, radii, cum, img_shape=img,
                                             block_width=BW)
    assert isect == ks.size and np.array_equal(gids, gs) and np.array_equal(bins, bs)
    assert np.array_equal(tids, ks >> 32)
