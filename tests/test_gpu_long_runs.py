"""Per-tile depth order of runs around and beyond what a workgroup holds (1536
entries for 256 threads, 3072 for the 512 threads that a second launch gives the
longer ones).

Views: the sorted ids must equal the oracle's (tile, depth bits, id) order
exactly, with few pairs per tile of the grid (the longer runs stay in the first
launch) and many (they go to the second).  Batches: the images must equal the
plain renders bit for bit.
"""

import numpy as np
import pytest

import oracle
from jaxsplat_amd import BatchPlan, ViewSpec, render, render_batch, scenes
from tests import helpers as H

pytestmark = pytest.mark.gpu

BW = 16


@pytest.mark.parametrize("rest", [3, 1500], ids=["one launch", "two"])
@pytest.mark.parametrize("ties", [1, 400])
def test_run_lengths(rest, ties):
    rng = np.random.default_rng(rest + ties)
    side = 17
    lengths = np.full(side * side, rest)
    edges = [0, 1, 2, 1535, 1536, 1537, 2047, 3071, 3072, 3073, 6000, 17000]
    lengths[rng.permutation(side * side)[:len(edges)]] = edges
    tile = rng.permutation(np.repeat(np.arange(side * side), lengths))
    n = tile.size
    # one tile each: a radius of a pixel about the tile's centre
    xys = (np.stack([tile % side, tile // side], 1) * BW + BW / 2).astype(np.float32)
    radii = np.ones(n, np.int32)
    bits = np.array(2.0, np.float32).view(np.uint32) + rng.integers(0, n // ties + 1, n)
    depths = bits.astype(np.uint32).view(np.float32)
    img = (side * BW, side * BW)
    cum = np.arange(1, n + 1, dtype=np.int32)
    gids, _, bins, isect = H.gpu_bin(xys, depths, radii, cum, img_shape=img, block_width=BW,
                                     rects=True)
    _, gs, bs = oracle.binning.bin_and_sort(xys, depths, radii, cum, img_shape=img,
                                            block_width=BW)
    assert isect == n and np.array_equal(np.diff(bins.reshape(-1, 2))[:, 0], lengths)
    assert np.array_equal(gids, gs)
    assert np.array_equal(bins, bs)


def test_batch_long_runs():
    t = H.torch()
    rng = np.random.default_rng(3)
    n, hw, f, c = 40000, (60, 76), (60.0, 60.0), (38.0, 30.0)
    p = [H.dev(a) for a in scenes.gaussians(rng, n, (-1.5, -1.2, 3), (1.5, 1.2, 6), np.log(0.05),
                                            opacity_logit_mean=-3.0)]
    vm = np.stack([scenes.IDENTITY, scenes.look_at((0.6, 0.2, -1.0), target=(0, 0, 4.5))])
    bg = H.dev(np.array([[0.1, 0.2, 0.3], [0.4, 0.5, 0.6]], np.float32))
    plan = BatchPlan([n], [ViewSpec(0, hw, f, c)] * 2, glob_scale=1.0, clip_thresh=0.01,
                     block_width=BW, isect_capacity=1 << 18)
    with t.no_grad():
        flat = render_batch(*p, H.dev(vm.astype(np.float32)), bg, plan=plan)
        assert plan.check() > 40 * 1537        # 20 tiles per view: runs beyond 1536
        for v, img in enumerate(plan.split(flat)):
            one = render(*p, viewmat=H.dev(vm[v].astype(np.float32)), background=bg[v],
                         img_shape=hw, f=f, c=c, glob_scale=1.0, clip_thresh=0.01, block_size=BW)
            assert np.array_equal(H.host(img), H.host(one))
