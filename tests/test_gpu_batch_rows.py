"""Batched binning by tile rows at the edges of its ranges: partitions of 1024
items, grids around 128 and 256 tiles per axis (257 takes the pair sort), views of
one Gaussian and views that see nothing, and a capacity one pair short.

Images must equal the plain renders bit for bit, and the gradients their sum over
a scene's views within 1e-3 |g| + 1e-4 max|g| (the order of the additions
differs); two runs bitwise identical.
"""

import numpy as np
import pytest

from jaxsplat_amd import BatchPlan, ViewSpec, _lib, render, render_batch, scenes
from tests import helpers as H

pytestmark = pytest.mark.gpu

SIZES = (1, 1023, 1025, 2600)           # Gaussians per scene
IMAGES = {4: [(60, 508), (508, 60), (77, 516), (516, 30)],      # up to 129 tiles
          8: [(300, 260), (40, 1027), (2048, 40), (90, 130)],     # up to 256
          5: [(33, 1281), (70, 60), (64, 200), (50, 50)],         # 257
          16: [(100, 90), (64, 64), (33, 47), (250, 300)]}


@pytest.mark.parametrize("bw", sorted(IMAGES))
def test_batch_rows(bw):
    t = H.torch()
    rng = np.random.default_rng(bw)
    n = sum(SIZES)
    params = [H.dev(a) for a in scenes.gaussians(rng, n, (-1.5, -1.2, 2), (1.5, 1.2, 6),
                                                 np.log(0.07))]
    away = scenes.look_at((0.0, 0.0, -30.0), target=(0.0, 0.0, -60.0))
    views, vms, first = [], [], np.cumsum((0,) + SIZES)
    for s, hw in enumerate(IMAGES[bw]):
        for vm in (scenes.IDENTITY, away if s == 1 else
                   scenes.look_at((0.5, 0.2, -1.0), target=(0, 0, 4))):
            f = float(max(hw)) * 0.8
            views.append(ViewSpec(s, hw, (f, f), (hw[1] / 2, hw[0] / 2)))
            vms.append(vm.astype(np.float32))
    vm = H.dev(np.stack(vms))
    bg = H.dev(rng.uniform(0, 1, (len(views), 3)).astype(np.float32))

    def plan(capacity):
        return BatchPlan(list(SIZES), views, glob_scale=1.0, clip_thresh=0.01, block_width=bw,
                         isect_capacity=capacity)

    pl = plan(1 << 19)
    runs = []
    for _ in range(2):
        p = [x.detach().clone().requires_grad_(True) for x in params]
        flat = render_batch(*p, vm, bg, plan=pl)
        v = t.linspace(-1, 1, flat.numel(), device="cuda").view(flat.shape)
        runs.append([flat.detach()] + list(t.autograd.grad(flat, p, v)))
    total = pl.check()
    for a, b in zip(*runs):
        assert np.array_equal(H.host(a).view(np.uint32), H.host(b).view(np.uint32))
    sums = [np.zeros(tuple(x.shape)) for x in params]
    for k, (img, vk) in enumerate(zip(pl.split(runs[0][0]), pl.split(v))):
        rows = slice(first[views[k].scene], first[views[k].scene + 1])
        p = [x[rows].detach().contiguous().requires_grad_(True) for x in params]
        one = render(*p, viewmat=vm[k].contiguous(), background=bg[k].contiguous(),
                     img_shape=tuple(img.shape[:2]), f=views[k].f, c=views[k].c, glob_scale=1.0,
                     clip_thresh=0.01, block_size=bw)
        assert np.array_equal(H.host(img).view(np.uint32), H.host(one.detach()).view(np.uint32))
        for s, g in zip(sums, t.autograd.grad(one, p, vk.contiguous())):
            s[rows] += H.host(g)
    for g, s in zip(runs[0][1:], sums):
        assert np.all(np.abs(H.host(g) - s) <= 1e-3 * np.abs(s) + 1e-4 * np.abs(s).max())

    short = plan(total - 1)
    with t.no_grad():
        render_batch(*params, vm, bg, plan=short)
    with pytest.raises(_lib.JaxsplatError):
        short.check()
    assert short.last_intersections == total
    exact = plan(total)
    with t.no_grad():
        again = render_batch(*params, vm, bg, plan=exact)
    assert exact.check() == total
    assert np.array_equal(H.host(again).view(np.uint32), H.host(runs[0][0]).view(np.uint32))


@pytest.mark.parametrize("adjoint", ["reference", "consistent"])
def test_batch_of_many_gaussians(adjoint):
    """With 131072 Gaussians or more the projection backward sums the records."""
    t = H.torch()
    rng = np.random.default_rng(9)
    sizes = (131072, 700)
    params = [H.dev(a) for a in scenes.gaussians(rng, sum(sizes), (-1.5, -1.2, 2),
                                                 (1.5, 1.2, 6), np.log(0.02))]
    hw, f, c = (120, 150), (120.0, 120.0), (75.0, 60.0)
    views = [ViewSpec(s, hw, f, c) for s in (0, 0, 1)]
    vms = [H.dev(scenes.look_at((x, 0.2, -1.0), target=(0, 0, 4)).astype(np.float32))
           for x in (0.5, -0.5, 0.0)]
    bg = H.dev(np.zeros((3, 3), np.float32))
    plan = BatchPlan(list(sizes), views, glob_scale=1.0, clip_thresh=0.01,
                     isect_capacity=1 << 20)
    runs = []
    for _ in range(2):
        p = [x.detach().clone().requires_grad_(True) for x in params]
        flat = render_batch(*p, t.stack(vms), bg, plan=plan, adjoint=adjoint)
        v = t.linspace(-1, 1, flat.numel(), device="cuda").view(flat.shape)
        runs.append(t.autograd.grad(flat, p, v))
    assert plan.check() > 0
    for a, b in zip(*runs):
        assert np.array_equal(H.host(a).view(np.uint32), H.host(b).view(np.uint32))
    sums = [np.zeros(tuple(x.shape)) for x in params]
    for k, vk in enumerate(plan.split(v)):
        rows = slice(0, sizes[0]) if k < 2 else slice(sizes[0], sum(sizes))
        p = [x[rows].detach().contiguous().requires_grad_(True) for x in params]
        one = render(*p, viewmat=vms[k], background=bg[k].contiguous(), img_shape=hw, f=f, c=c,
                     glob_scale=1.0, clip_thresh=0.01, adjoint=adjoint)
        for s, g in zip(sums, t.autograd.grad(one, p, vk.contiguous())):
            s[rows] += H.host(g)
    for g, s in zip(runs[0], sums):
        assert np.all(np.abs(H.host(g) - s) <= 1e-3 * np.abs(s) + 1e-4 * np.abs(s).max())
