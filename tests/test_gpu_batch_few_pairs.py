"""Batches on both sides of the rule that takes few pairs to the pair sort instead of
the binning by tile rows: views of up to 64 tiles, of up to 256 tiles with a capacity
around 1M, and few items in flat views with a capacity around 2.5M.

Images must equal the plain renders bit for bit, and images, gradients and totals of
the two sides each other.
"""

import numpy as np
import pytest

from jaxsplat_amd import BatchPlan, ViewSpec, _lib, render, render_batch, scenes
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _bits(x):
    return H.host(x).view(np.uint32)


@pytest.mark.parametrize("shapes,n,caps", [
    ([(64, 100), (17, 33)], 900, (100_000, 3_000_000)),
    ([(128, 129), (17, 250), (256, 256)], 900, (999_999, 1_000_000)),
    ([(60, 1000), (100, 1500)], 1500, (2_499_999, 2_500_000)),
    ([(1000, 60)], 1500, (2_499_999, 2_500_000))], ids=str)
def test_both_sides_agree(shapes, n, caps):
    t = H.torch()
    rng = np.random.default_rng(n + len(shapes))
    params = [H.dev(a) for a in scenes.gaussians(rng, n, (-1.5, -1.2, 2), (1.5, 1.2, 6),
                                                 np.log(0.15))]
    views = [ViewSpec(0, hw, (float(max(hw)),) * 2, (hw[1] / 2, hw[0] / 2)) for hw in shapes * 2]
    vms = H.dev(np.stack([scenes.look_at((0.5 * np.sin(k), 0.2, -1.0), target=(0, 0, 4))
                          for k in range(len(views))]).astype(np.float32))
    bg = H.dev(rng.uniform(0, 1, (len(views), 3)).astype(np.float32))
    runs = []
    for cap in caps:
        plan = BatchPlan([n], views, glob_scale=1.0, clip_thresh=0.01, isect_capacity=cap)
        p = [x.detach().clone().requires_grad_(True) for x in params]
        flat = render_batch(*p, vms, bg, plan=plan)
        v = t.linspace(-1, 1, flat.numel(), device="cuda").view(flat.shape)
        grads = t.autograd.grad(flat, p, v)
        runs.append(([flat.detach(), *grads], plan.check()))
    assert runs[0][1] == runs[1][1] > 1000
    assert all(np.array_equal(_bits(a), _bits(b)) for a, b in zip(runs[0][0], runs[1][0]))
    for k, img in enumerate(plan.split(runs[0][0][0])):
        hw = views[k].img_shape
        one = render(*params, viewmat=vms[k].contiguous(), background=bg[k].contiguous(),
                     img_shape=hw, f=views[k].f, c=views[k].c, glob_scale=1.0, clip_thresh=0.01)
        assert np.array_equal(_bits(img), _bits(one)), k
    short = BatchPlan([n], views, glob_scale=1.0, clip_thresh=0.01, isect_capacity=runs[0][1] - 1)
    with t.no_grad():
        render_batch(*params, vms, bg, plan=short)
    with pytest.raises(_lib.JaxsplatError):
        short.check()
    assert short.last_intersections == runs[0][1]
