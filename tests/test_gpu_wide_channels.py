"""More than three channels: passes of up to eight channels over one list.

The image must be bit for bit that of three-channel renders of the same
channels (every pass takes the same blend decisions), and the gradients those of
the atomic backward's three-channel passes on the same lists.  Bar 1e-4 |g| +
2e-5 max|g|: a pass of eight channels carries one sum of what lies behind for
all of its channels where three passes carry one each, over lists of up to ~100
blending entries (100 roundings of 6e-8 of terms that may cancel by a few
times).  Two runs bitwise identical.
"""

import numpy as np
import pytest

from jaxsplat_amd import _ops, project, rasterize, scenes
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nch,block,adjoint,tight", [
    (4, 16, "reference", True), (5, 16, "consistent", True), (7, 8, "reference", False),
    (8, 16, "reference", False), (9, 12, "consistent", True), (12, 8, "consistent", False),
    (20, 16, "reference", True), (4, 4, "consistent", True)])
def test_wide_channels(nch, block, adjoint, tight, monkeypatch):
    t = H.torch()
    monkeypatch.setattr(_ops, "TIGHT_TILES", tight)
    rng = np.random.default_rng(23)
    n, size = 3000, (100, 141)
    means = np.concatenate([rng.uniform(-2, 2, (n, 2)), rng.uniform(3, 6, (n, 1))], 1)
    scales = np.exp(rng.normal(np.log(0.06), 0.5, (n, 3)))
    quats = rng.normal(size=(n, 4))
    quats /= np.linalg.norm(quats, axis=1, keepdims=True)
    with t.no_grad():
        out = project(*[H.dev(a.astype(np.float32)) for a in (means, scales, quats)],
                      H.dev(scenes.IDENTITY), img_shape=size, f=(140.0, 140.0),
                      c=(70.0, 50.0), glob_scale=1.0, clip_thresh=0.01, block_width=block)
    xys, depths, radii, conics, _, cum = out
    opac = H.dev(rng.uniform(0.05, 0.95, (n, 1)).astype(np.float32))
    colors = H.dev(rng.uniform(0, 1, (n, nch)).astype(np.float32))
    bg = H.dev(rng.uniform(0, 1, nch).astype(np.float32))
    v = H.dev(rng.normal(size=(*size, nch)).astype(np.float32))
    kw = dict(img_shape=size, block_width=block)

    def render(col, back, leaves):
        return rasterize(col, leaves[0], back, leaves[1], depths, radii, leaves[2], cum,
                         adjoint=adjoint, **kw)

    runs = []
    for staged in (True, True, False):
        monkeypatch.setattr(_ops, "STAGED_BACKWARD", staged)
        leaves = [x.detach().clone().requires_grad_(True) for x in (colors, opac, xys, conics)]
        img = render(leaves[0], bg, leaves[1:])
        runs.append([H.host(img.detach())] + [H.host(g) for g in t.autograd.grad(img, leaves, v)])
    with t.no_grad():
        for k in range(0, nch, 3):
            part = render(colors[:, k:k + 3].contiguous(), bg[k:k + 3].contiguous(),
                          (opac, xys, conics))
            assert np.array_equal(runs[0][0][..., k:k + 3].view(np.uint32),
                                  H.host(part).view(np.uint32))
    for a, b, c in zip(*runs):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        ref = c.astype(np.float64)
        assert np.abs(ref).max() > 0
        assert np.all(np.abs(a - ref) <= 1e-4 * np.abs(ref) + 2e-5 * np.abs(ref).max())
