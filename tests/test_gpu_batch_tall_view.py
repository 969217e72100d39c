"""A batch of many small views with one of 256 tile rows between them: workspace by
the tile rows that the views have, and the images of the views bit for bit the
plain renders'."""

import numpy as np
import pytest

from jaxsplat_amd import BatchPlan, ViewSpec, render, render_batch, scenes
from tests import helpers as H

pytestmark = pytest.mark.gpu

N, SMALL, CAP = 300, 1000, 1 << 20


def _views(shapes):
    return [ViewSpec(0, hw, (float(max(hw)),) * 2, (hw[1] / 2, hw[0] / 2)) for hw in shapes]


def _plan(shapes):
    return BatchPlan([N], _views(shapes), glob_scale=1.0, clip_thresh=0.01, isect_capacity=CAP)


def test_one_tall_view_among_many():
    t = H.torch()
    rng = np.random.default_rng(4)
    params = [H.dev(a) for a in scenes.gaussians(rng, N, (-1.5, -1.2, 2), (1.5, 1.2, 6),
                                                 np.log(0.07))]
    shapes = [(32, 20 + k % 13) for k in range(SMALL // 2)]
    shapes = shapes + [(4096, 32)] + shapes
    vms = np.stack([scenes.look_at((0.5 * np.sin(k), 0.2, -1.0), target=(0, 0, 4))
                    for k in range(len(shapes))]).astype(np.float32)
    vm, bg = H.dev(vms), t.full((len(shapes), 3), 0.25, device="cuda")

    plan = _plan(shapes)
    # the tables of the views' tile rows add up (the bins, 8 bytes each, are padded to
    # the largest view)
    small, tall = _plan([(32, 32)] * len(shapes)), _plan([(4096, 32)])
    assert plan.workspace_bytes <= \
        small.workspace_bytes + tall.workspace_bytes + 8 * 1024 * len(shapes)

    p = [x.detach().clone().requires_grad_(True) for x in params]
    flat = render_batch(*p, vm, bg, plan=plan)
    assert plan.check() > 10_000
    images = plan.split(flat.detach())
    for k in [0, 1, 499, 500, 501, 777, 1000]:
        hw = shapes[k]
        one = render(*params, viewmat=vm[k].contiguous(), background=bg[k].contiguous(),
                     img_shape=hw, f=(float(max(hw)),) * 2, c=(hw[1] / 2, hw[0] / 2),
                     glob_scale=1.0, clip_thresh=0.01)
        assert np.array_equal(H.host(images[k]).view(np.uint32), H.host(one).view(np.uint32)), k
    grads = t.autograd.grad(flat, p, t.ones_like(flat))
    assert all(bool(t.isfinite(g).all()) for g in grads)
