"""Binning into a capacity below the intersection count: the pairs that are binned
are the first ``capacity`` of the emission order (Gaussian by Gaussian, each
rectangle row by row; reference ``lib/kernels/forward.cu:135-179``), sorted as
always, with bit 8 of the error word and the exact total in the workspace's header.

Sorted ids, tile ids and bins must equal the oracle's order of those pairs exactly,
at capacities that end between two Gaussians, after a whole row of a rectangle and
inside one: for the pair sort (few Gaussians over many tiles), by rows in id order and
in depth order (65600 Gaussians, 0.06 of them over the whole grid), and where 128 and 256 tiles per
axis change the kernels.
"""

import ctypes

import numpy as np
import pytest

import oracle
from jaxsplat_amd import _lib
from tests import helpers as H

pytestmark = pytest.mark.gpu

BW = 16


def _scene(n, tiles, whole, seed):
    rng = np.random.default_rng(seed)
    h, w = tiles[0] * BW - 3, tiles[1] * BW - 5
    xys = np.stack([rng.uniform(-10, w + 10, n), rng.uniform(-10, h + 10, n)], 1).astype(np.float32)
    radii = rng.integers(1, 60 if n < 10000 else 12, n).astype(np.int32)
    radii[rng.random(n) < 0.1] = 0
    radii[rng.random(n) < whole] = max(h, w) + 20
    bits = np.array(2.0, np.float32).view(np.uint32) + rng.integers(0, max(n // 4, 1), n)
    depths = bits.astype(np.uint32).view(np.float32)
    x0, x1, y0, y1 = oracle.project.tile_rect(xys[:, 0], xys[:, 1], radii.astype(np.float32),
                                              tiles[1], tiles[0], BW)
    on = radii > 0
    width = np.where(on, x1 - x0, 0)
    cum = np.cumsum(np.where(on, width * (y1 - y0), 0)).astype(np.int32)
    return xys, depths, radii, cum, width, (h, w)


def _bin(path, xys, depths, radii, cum, img, cap):
    """(ids, tile ids, bins, error word, exact total) of one binning call."""
    t, L = H.torch(), _lib.lib()
    d = H.descriptor(xys.shape[0], img, block_width=BW)
    D = ctypes.byref(d)
    x, dp, r = H.dev(xys), H.dev(depths), H.dev(radii)
    gids, tids = (t.full((cap,), -5, dtype=t.int32, device="cuda") for _ in range(2))
    bins = t.full((d.grid_dim_2d.x * d.grid_dim_2d.y, 2), -5, dtype=t.int32, device="cuda")
    out = [H.P(gids), H.P(tids), H.P(bins)]

    def buffer(size):
        return t.full((max(size, 16),), 0xA5, dtype=t.uint8, device="cuda")

    if path == "one":
        ws = buffer(L.jaxsplat_bin_workspace_size(D, cap))
        _lib.check(L.jaxsplat_bin_and_sort(D, H.P(x), H.P(dp), H.P(r), cap, *out, H.P(ws),
                                           ws.numel(), H.stream()))
    elif path == "split":
        dws = buffer(L.jaxsplat_bin_depth_workspace_size(D))
        ws = buffer(L.jaxsplat_bin_emit_workspace_size(D, cap))
        _lib.check(L.jaxsplat_bin_depth_sort(D, H.P(x), H.P(dp), H.P(r), H.P(dws), dws.numel(),
                                             H.stream()))
        _lib.check(L.jaxsplat_bin_emit_sort(D, cap, H.P(dws), *out, H.P(ws), ws.numel(),
                                            H.stream()))
    else:
        rc, cm = H.dev(H.packed_rects(xys, radii, img, BW)), H.dev(cum)
        ws = buffer(L.jaxsplat_bin_emit_workspace_size(D, cap))
        _lib.check(L.jaxsplat_bin_rects_sort(D, H.P(dp), H.P(rc), H.P(cm), cap, *out, H.P(ws),
                                             ws.numel(), H.stream()))
    header = H.host(ws[:16])
    return (H.host(gids), H.host(tids), H.host(bins), int(header[:4].view(np.uint32)[0]),
            int(header[8:].view(np.uint64)[0]))


@pytest.mark.parametrize("path", ["one", "split", "rects"])
@pytest.mark.parametrize("n,tiles,whole", [
    (700, (9, 9), 0.05), (1500, (17, 17), 0.05), (2600, (30, 20), 0.01), (2100, (3, 129), 0.02),
    (2100, (129, 3), 0.02), (1200, (2, 256), 0.05), (1200, (256, 2), 0.05), (900, (2, 257), 0.05),
    (1700, (17, 17), 0.6), (65600, (17, 17), 0.002), (65600, (17, 17), 0.06),
    (65600, (129, 4), 0.001), (65600, (4, 129), 0.001)], ids=str)
def test_first_pairs_of_the_emission_order(n, tiles, whole, path):
    xys, depths, radii, cum, width, img = _scene(n, tiles, whole, seed=n + tiles[0])
    total = int(cum[-1])
    keys, gids = oracle.binning.emit(xys, depths, radii, cum, img_shape=img, block_width=BW)
    # a wide rectangle in the last tenth, so that the depth order stays chosen
    g = int(n - n // 10 + np.argmax(width[n - n // 10:]))
    first, w = int(cum[g - 1]), int(width[g])
    assert w > 1
    for cap in (total + 5, total, total - 1, first, first + w, first + w + 1, first + 1,
                total // 3, 1):
        ids, tids, bins, err, exact = _bin(path, xys, depths, radii, cum, img, cap)
        m = min(total, cap)
        ks, gs = oracle.binning.sort_pairs(keys[:m], gids[:m], tiles[0] * tiles[1])
        assert exact == total and err == (8 if total > cap else 0), cap
        assert np.array_equal(ids[:m], gs), cap
        assert np.array_equal(tids[:m], ks >> 32), cap
        assert np.array_equal(bins, oracle.binning.tile_bins(ks, tiles[0] * tiles[1])), cap
