"""Sums of the staged backward's records (``sum_records``) over ranges of few
and many slots, with few and many of them flagged.

A Gaussian's records are summed by its own lane (at most 16 slots, or at most
two flagged), or by the whole wave (more, and ranges of more bitmap words than a
lane counts).  Bar, as for the staged backward: within 1e-5 |g| + 1e-6 max|g| of
the atomic backward on the same lists (only the order of the additions differs);
two runs bitwise identical.
"""

import numpy as np
import pytest

from jaxsplat_amd import _ops, project, rasterize, scenes
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,scale,thin,opaque", [
    ((256, 256), 0.05, 1.0, False),         # a few slots per Gaussian
    ((480, 640), 0.6, 1.0, False),          # hundreds, most of them flagged
    ((480, 640), 0.6, 1.0, True),           # hundreds, few flagged behind the front ones
    ((1040, 1040), 2.5, 0.02, False),       # diagonals: thousands of slots, few flagged
], ids=["narrow", "many", "opaque", "wide"])
def test_record_sums(size, scale, thin, opaque, monkeypatch):
    t = H.torch()
    rng = np.random.default_rng(17)
    n = 400
    h, w = size
    means = np.concatenate([rng.uniform(-2, 2, (n, 2)), rng.uniform(4, 6, (n, 1))], 1)
    scales = np.stack([np.full(n, scale), np.full(n, scale * thin), np.full(n, scale * thin)], 1)
    quats = rng.normal(size=(n, 4))
    if thin < 1:                            # turned about the view axis only
        quats[:, 1:3] = 0
    quats /= np.linalg.norm(quats, axis=1, keepdims=True)
    opac = H.dev((rng.uniform(0.9, 0.98, (n, 1)) if opaque else
                  rng.uniform(0.02, 0.4, (n, 1))).astype(np.float32))
    with t.no_grad():
        out = project(*[H.dev(a.astype(np.float32)) for a in (means, scales, quats)],
                      H.dev(scenes.IDENTITY), img_shape=size, f=(float(w), float(w)),
                      c=(w / 2, h / 2), glob_scale=1.0, clip_thresh=0.01, block_width=16)
    xys, depths, radii, conics, _, cum = out
    colors = H.dev(rng.uniform(0, 1, (n, 3)).astype(np.float32))
    v = H.dev(rng.normal(size=(*size, 3)).astype(np.float32))
    runs = []
    for staged in (True, True, False):
        monkeypatch.setattr(_ops, "STAGED_BACKWARD", staged)
        leaves = [x.detach().clone().requires_grad_(True) for x in (colors, opac, xys, conics)]
        img = rasterize(leaves[0], leaves[1], t.zeros(3, device="cuda"), leaves[2], depths, radii,
                        leaves[3], cum, img_shape=size, block_width=16)
        runs.append([H.host(g) for g in t.autograd.grad(img, leaves, v)])
    for a, b, c in zip(*runs):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        ref = c.astype(np.float64)
        assert np.abs(ref).max() > 0
        assert np.all(np.abs(a - ref) <= 1e-5 * np.abs(ref) + 1e-6 * np.abs(ref).max())
