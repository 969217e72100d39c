"""A capacity's headroom must not choose how the lists are ordered: as many kernels
for a generous capacity as for a tight one (but for the second launch for long
runs), fewer than the depth sort of the Gaussians takes; with the total that
``check()`` read, the kernels that the total calls for, whatever the capacity.
Images bit for bit the same throughout."""

import ctypes

import numpy as np
import pytest

from jaxsplat_amd import IsectCapacity, _lib, _ops, render, scenes
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _kernels(fn):
    """Nodes of the graph that captures fn, and fn's result from a replay."""
    t = H.torch()
    side = t.cuda.Stream()
    side.wait_stream(t.cuda.current_stream())
    with t.cuda.stream(side):
        fn()
    t.cuda.current_stream().wait_stream(side)
    t.cuda.synchronize()
    g = t.cuda.CUDAGraph(keep_graph=True)
    with t.cuda.graph(g):
        out = fn()
    n = ctypes.c_size_t()
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    g.replay()
    return n.value, H.host(out)


def _scene(n, log_scale, size, channels):
    t = H.torch()
    rng = np.random.default_rng(n)
    p = [H.dev(a) for a in scenes.gaussians(rng, n, (-2, -1.5, 2), (2, 1.5, 6), log_scale)]
    p[3] = p[3][:, :1].repeat(1, channels).contiguous()
    kw = dict(viewmat=H.dev(scenes.IDENTITY), background=t.zeros(channels, device="cuda"),
              img_shape=size, f=(float(size[1]),) * 2, c=(size[1] / 2, size[0] / 2),
              glob_scale=1.0, clip_thresh=0.01)

    def run(cap=None):
        with t.no_grad():
            return render(*p, **kw, isect_capacity=cap)

    return run


# the fused render, its two-stage binning on the reference's rectangles, and separate
# nodes of more than three channels
PATHS = {"fused": (3, True), "reference tiles": (3, False), "wide": (5, True)}


@pytest.mark.parametrize("path", sorted(PATHS))
def test_headroom_adds_no_depth_sort(path, monkeypatch):
    channels, tight = PATHS[path]
    monkeypatch.setattr(_ops, "TIGHT_TILES", tight)
    run = _scene(70000, np.log(0.01), (330, 400), channels)    # 525 tiles, short lists
    probe = IsectCapacity(1 << 22)
    want = H.host(run(probe))
    total = probe.check()
    assert total < 640 * 525
    tight_cap = IsectCapacity(total)
    base, img = _kernels(lambda: run(tight_cap))
    assert np.array_equal(img, want)
    for cap in (1 << 21, 1 << 24):
        known = IsectCapacity(cap)
        nodes, img = _kernels(lambda: run(known))
        assert np.array_equal(img, want)
        assert nodes <= base + 1, cap
        assert known.check() == total
        nodes, img = _kernels(lambda: run(known))
        assert np.array_equal(img, want)
        assert nodes == base, cap


@pytest.mark.parametrize("path", sorted(PATHS))
def test_checked_total_chooses_the_depth_order(path, monkeypatch):
    channels, tight = PATHS[path]
    monkeypatch.setattr(_ops, "TIGHT_TILES", tight)
    run = _scene(6000, np.log(0.6), (330, 400), channels)      # large ones: long lists
    want = H.host(run())
    cap = IsectCapacity(1 << 23)
    unknown, img = _kernels(lambda: run(cap))
    assert np.array_equal(img, want)
    total = cap.check()
    assert total > 1_000_000
    nodes, img = _kernels(lambda: run(cap))
    assert np.array_equal(img, want)
    assert nodes > unknown + 3
    cap.check()
    cap.check()                                 # nothing rendered: still known
    assert _kernels(lambda: run(cap))[0] == nodes


def test_few_pairs_are_not_sorted_by_depth():
    """Long lists of few pairs (fewer than 0.75M): hardly more kernels than short lists of
    as many Gaussians (a depth sort of them is eight)."""
    nodes = []
    for log_scale in (np.log(0.01), np.log(0.6)):
        run = _scene(3000, log_scale, (272, 272), 3)           # 289 tiles
        want = H.host(run())
        cap = IsectCapacity(1 << 22)
        run(cap)
        total = cap.check()
        tight = IsectCapacity(total)
        run(tight)
        assert tight.check() == total
        n, img = _kernels(lambda: run(tight))
        assert np.array_equal(img, want)
        nodes.append(n)
    assert 16 * 3000 < total < 750_000 and total > 640 * 289
    assert nodes[1] <= nodes[0] + 5
