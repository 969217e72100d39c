"""Which binning a view takes depends on its Gaussians and its capacity: few Gaussians
with many pairs each take the pair sort up to 4M pairs, others tile rows.  With a
capacity of 4M the scenes of ``test_gpu_row_bin`` are binned by rows whatever their
size, and at the limits of the rule the scenes here take either.

Sorted ids, tile ids and bins must equal the oracle's stable (tile, depth bits, id)
order exactly, on the edges of partitions (1023, 1025 Gaussians), of the LDS widths
(128 and 256 tiles per axis), with rectangles over the whole grid, with the lists
ordered tile by tile (expected 0) and by one depth sort (expected 4M).
"""

import ctypes

import numpy as np
import pytest

import oracle
from jaxsplat_amd import _lib
from tests import helpers as H
from tests import test_gpu_row_bin as R

pytestmark = pytest.mark.gpu

CAP = 4_000_001


def _check(scene, tiles, cap, expected, path):
    xys, depths, radii, cum, img = scene
    t, L, n = H.torch(), _lib.lib(), xys.shape[0]
    D = ctypes.byref(H.descriptor(n, img, block_width=R.BW))
    x, dp, r = H.dev(xys), H.dev(depths), H.dev(radii)
    gids, tids = (t.full((cap,), -5, dtype=t.int32, device="cuda") for _ in range(2))
    bins = t.full((tiles[0] * tiles[1], 2), -5, dtype=t.int32, device="cuda")
    out = [H.P(gids), H.P(tids), H.P(bins)]
    ws = t.full((L.jaxsplat_bin_emit_workspace_size(D, cap),), 0xA5, dtype=t.uint8, device="cuda")
    if path == "rects":
        rc, cm = H.dev(H.packed_rects(xys, radii, img, R.BW)), H.dev(cum)
        _lib.check(L.jaxsplat_bin_rects_sort_expecting(D, H.P(dp), H.P(rc), H.P(cm), cap, expected,
                                                       *out, H.P(ws), ws.numel(), H.stream()))
    else:
        size = L.jaxsplat_bin_depth_workspace_size(D)
        dws = t.full((size,), 0xA5, dtype=t.uint8, device="cuda")
        _lib.check(L.jaxsplat_bin_depth_sort(D, H.P(x), H.P(dp), H.P(r), H.P(dws), size,
                                             H.stream()))
        _lib.check(L.jaxsplat_bin_emit_sort_expecting(D, cap, expected, H.P(dws), *out, H.P(ws),
                                                      ws.numel(), H.stream()))
    ks, gs, bs = oracle.binning.bin_and_sort(xys, depths, radii, cum, img_shape=img,
                                             block_width=R.BW)
    m = min(cap, ks.size)
    header = H.host(ws[:16])
    assert int(header[8:].view(np.uint64)[0]) == ks.size and header[:4].view(np.uint32)[0] == 0
    assert m == ks.size
    assert np.array_equal(H.host(gids)[:m], gs)
    assert np.array_equal(H.host(tids)[:m], ks >> 32)
    assert np.array_equal(H.host(bins), bs)
    assert np.all(H.host(gids)[m:] == -5)       # nothing behind the pairs


GRIDS = [(17, 17), (128, 3), (129, 3), (3, 128), (3, 129), (2, 256), (256, 2)]


@pytest.mark.parametrize("path", ["split", "rects"])
@pytest.mark.parametrize("expected", [0, CAP], ids=["tile by tile", "by depth"])
@pytest.mark.parametrize("n", [1, 1023, 1025, 6000])
@pytest.mark.parametrize("tiles", GRIDS, ids=str)
def test_rows_by_capacity(tiles, n, expected, path):
    for radius in (12, 90):
        scene = R._scene(n, tiles, radius, seed=n + radius + tiles[0])
        if scene[3][-1] == 0:
            continue
        _check(scene, tiles, CAP, expected, path)


@pytest.mark.parametrize("path", ["split", "rects"])
@pytest.mark.parametrize("n,tiles,cap", [
    (12287, (20, 20), 48 * 12287), (12287, (20, 20), 48 * 12287 + 1),
    (32767, (8, 40), 16 * 32767), (32767, (8, 40), 16 * 32767 + 1),
    (12287, (20, 20), 3_999_999), (12287, (20, 20), 4_000_000), (12288, (20, 20), 400_000),
    (32767, (8, 40), 3_999_999), (32767, (40, 8), 4_000_000), (32768, (8, 40), 400_000),
    (32767, (9, 40), 400_000)],
    ids=str)
def test_limits_of_the_rule(n, tiles, cap, path):
    _check(R._scene(n, tiles, 12, seed=n), tiles, cap, 0, path)
