"""Performance cases of jaxsplat_amd: what its users have it do, with seeded inputs.

Every case renders synthetic scenes of the kinds that the tests and ``bench.py`` use:

* ``"volume"``  -- Gaussians in a box before the camera that is a little wider than its view (the ``small``,
  ``hd1m`` and ``dense3m`` workloads of ``jaxsplat_amd.scenes``): ``log_scale`` is the mean of the world scales' log,
  ``logit`` the mean of the opacities' logits.
* ``"random"``  -- the reference benchmark's parameters (``examples/benchmark.py:236-279``): Gaussians of up to half a
  unit in a cube 8 units away, each over many tiles.
* ``"orbit"``   -- a cube of Gaussians seen by cameras around it (the ``orbit64`` workload).

A case's ``call`` says how the program calls the framework:

* ``"view"``  -- one forward ``render`` without gradients: a viewer, an evaluation;
* ``"step"``  -- ``render`` and the gradients of its five inputs for a given image cotangent: a training step;
* ``"ops"``   -- the same with ``project`` and ``rasterize`` called one after the other;
* ``"batch"`` -- ``render_batch`` over all views of a plan, and its gradients.

``exact`` restates the forward and the reference's adjoint in torch float64.
"""

import math

import torch

import jaxsplat_amd

_PARAMS = ("means3d", "scales", "quats", "colors", "opacities")
_CLIP = 0.01


def _case(name, call, scene, n, h, w, **more):
    c = {"call": call, "scene": scene, "n": n, "h": h, "w": w, "channels": 3, "block": 16,
         "log_scale": math.log(0.02), "logit": 0.0, "adjoint": "reference", "antialiased": False,
         "capacity": False, "views": 1, "scenes": 1}
    c.update(more)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: a preview of a small model, where launches and host work are all there is
        _case("view_2k_256", "view", "volume", 2_000, 256, 256, log_scale=math.log(0.08)),
        # the smallest training step (the `small` workload's sizes)
        _case("step_10k_256", "step", "volume", 10_000, 256, 256, log_scale=math.log(0.05)),
        # the reference's own benchmark: 50k Gaussians, 1600 x 900, forward, white background
        _case("view_50k_1600x900", "view", "random", 50_000, 900, 1600),
        # fitting Gaussians to one picture from a random start (the reference's training example), with a
        # fixed intersection capacity so that the loop never waits for the GPU; an odd picture size
        _case("step_fit_50k_1021x683", "step", "random", 50_000, 683, 1021, capacity=True),
        # the headline training step: 1M Gaussians at 1080p
        _case("step_1m_1080p", "step", "volume", 1_000_000, 1080, 1920),
        # the same with a fixed capacity, as a loop that never reads back a count runs it, at an uneven size
        _case("step_610k_1080p_capacity", "step", "volume", 610_007, 1080, 1920, capacity=True,
              log_scale=math.log(0.03)),
        # deep tile lists: 3M large, nearly opaque Gaussians (the `dense3m` workload)
        _case("step_dense_3m_1080p", "step", "volume", 3_000_000, 1080, 1920,
              log_scale=math.log(0.05), logit=4.0),
        # a large model shown on a 4K screen
        _case("view_2m_2160p", "view", "volume", 2_000_000, 2160, 3840),
        # the antialiased mode, at a ragged picture size, with the exact adjoint
        _case("step_antialiased_300k_719p", "step", "volume", 300_000, 719, 1277, antialiased=True,
              adjoint="consistent"),
        # feature rendering: 7 channels per Gaussian
        _case("step_7ch_200k_540p", "step", "volume", 200_001, 540, 960, channels=7),
        # project and rasterize called separately, on the smaller tiles
        _case("ops_block8_100k_512", "ops", "volume", 100_000, 512, 512, block=8),
        # multi-view training: 12 cameras around one scene in one call
        _case("batch_12x800_500k", "batch", "orbit", 500_000, 800, 800, views=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(("view", "view", "step", "step", "step", "ops", "batch"))
    if call == "batch":
        views = rng.randint(2, 12)
        side = _log_int(rng, 200, 800)
        scenes = rng.choice((1, 1, 2, 3))
        return _case(None, call, "orbit", _log_int(rng, 10_000, 400_000) // scenes, side,
                     _log_int(rng, 200, 800), views=views, scenes=min(scenes, views))
    scene = rng.choice(("volume", "volume", "volume", "random"))
    most = (2160, 3840) if call == "view" and scene == "volume" else (1080, 1920)
    h = _log_int(rng, 200, most[0])
    w = min(most[1], max(200, int(h * rng.uniform(1.0, 1.9))))
    more = {}
    if scene == "random":
        n = _log_int(rng, 2_000, 60_000)
    else:
        n = _log_int(rng, 2_000, 1_500_000)
        # larger Gaussians for smaller models: the scene stays covered
        more["log_scale"] = math.log(rng.uniform(0.01, 0.03) * (1e6 / max(n, 30_000)) ** 0.25)
        more["logit"] = rng.choice((0.0, 0.0, 2.0))
    if call == "step":
        option = rng.choice(("plain", "plain", "capacity", "antialiased", "channels"))
        more["capacity"] = option == "capacity"
        more["antialiased"] = option == "antialiased"
        if option == "channels":
            more["channels"] = rng.randint(1, 8)
            n = min(n, 300_000)
    if call != "view":
        more["adjoint"] = rng.choice(("reference", "reference", "consistent"))
    # the small tiles go with small pictures
    more["block"] = rng.choice((16, 8)) if h * w < 500_000 else 16
    return _case(None, call, scene, n, h, w, **more)


# -- inputs -------------------------------------------------------------------

def _gaussians(case, gen, dev):
    """The scene's parameters: means3d, scales, quats, colors, opacities, on `dev` in float32."""
    n = case["n"] * case["scenes"]

    def u(k, lo, hi):
        return torch.rand((n, k), generator=gen, device=dev) * (hi - lo) + lo

    def normal(k):
        return torch.randn((n, k), generator=gen, device=dev)

    if case["scene"] == "random":
        means, scales = u(3, -3.0, 3.0), u(3, 0.0, 0.5)
    else:
        if case["scene"] == "orbit":
            means = u(3, -2.0, 2.0)
        else:
            aspect = case["h"] / case["w"]
            means = torch.cat([u(1, -4.0, 4.0), u(1, -4.4 * aspect, 4.4 * aspect), u(1, 2.0, 10.0)], 1)
        scales = torch.exp(normal(3) * 0.3 + case["log_scale"])
    quats = torch.nn.functional.normalize(normal(4), dim=1)
    colors = u(case["channels"], 0.0, 1.0)
    opacities = u(1, 0.0, 1.0) if case["scene"] == "random" \
        else torch.sigmoid(normal(1) * (0.5 if case["logit"] >= 4 else 1.0) + case["logit"])
    return [means, scales, quats, colors, opacities]


def _cameras(case, gen, dev):
    """viewmats (V, 4, 4), the focal lengths and the principal point."""
    h, w, views = case["h"], case["w"], case["views"]
    vm = torch.eye(4, device=dev).repeat(views, 1, 1)
    if case["scene"] == "random":
        vm[:, 2, 3] = 8.0
        f = (w / 2, h / 2)
    elif case["scene"] == "volume":
        f = (w * 0.78, w * 0.78)
    else:
        az = torch.rand(views, generator=gen, device=dev) * (2 * math.pi)
        el = (torch.rand(views, generator=gen, device=dev) - 0.5) * (math.pi / 3)
        eye = 8.0 * torch.stack([el.cos() * az.sin(), el.sin(), el.cos() * az.cos()], 1)
        fwd = -eye / eye.norm(dim=1, keepdim=True)
        up = torch.tensor([0.0, 1.0, 0.0], device=dev).expand(views, 3)
        right = torch.nn.functional.normalize(torch.linalg.cross(up, fwd), dim=1)
        vm[:, :3, :3] = torch.stack([right, torch.linalg.cross(fwd, right), fwd], 1)
        vm[:, :3, 3] = -(vm[:, :3, :3] @ eye[:, :, None])[:, :, 0]
        f = (float(max(h, w)), float(max(h, w)))
    return vm, f, (w / 2, h / 2)


def _inputs(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    params = _gaussians(case, gen, dev)
    viewmats, f, c = _cameras(case, gen, dev)
    ch, pixels = case["channels"], case["h"] * case["w"] * case["views"]
    back = torch.ones if case["scene"] == "random" else torch.zeros
    backgrounds = back((case["views"], ch), device=dev)
    # the gradient of an L2 loss between two unlike pictures
    v_img = None
    if case["call"] != "view":
        v_img = torch.rand((pixels, ch), generator=gen, device=dev)
        v_img.sub_(torch.rand((pixels, ch), generator=gen, device=dev)).mul_(2.0 / (pixels * ch))
        if case["call"] != "batch":
            v_img = v_img.view(case["h"], case["w"], ch)
    return params, viewmats, backgrounds, f, c, v_img


def _view_scene(case, v):
    """The scene that view v looks at (views are grouped by scene)."""
    return v * case["scenes"] // case["views"]


def prepare(case, seed):
    params, viewmats, backgrounds, f, c, v_img = _inputs(case, seed)
    state = {"case": case, "v_img": v_img, "viewmats": viewmats, "backgrounds": backgrounds}
    if case["call"] != "view":
        for p in params:
            p.requires_grad_(True)
    state["params"] = params
    size = (case["h"], case["w"])
    if case["call"] == "batch":
        views = [jaxsplat_amd.ViewSpec(_view_scene(case, v), size, f, c) for v in range(case["views"])]
        renderer = jaxsplat_amd.BatchRenderer([case["n"]] * case["scenes"], views, clip_thresh=_CLIP,
                                              block_width=case["block"], check_every=0)
        with torch.no_grad():           # the first call sizes the plan
            renderer(*params, viewmats, backgrounds, adjoint=case["adjoint"])
        state["renderer"] = renderer
        return state
    state["camera"] = {"viewmat": viewmats[0].contiguous(), "img_shape": size, "f": f, "c": c,
                       "glob_scale": 1.0, "clip_thresh": _CLIP}
    state["background"] = backgrounds[0].contiguous()
    state["capacity"] = None
    if case["capacity"]:
        cap = jaxsplat_amd.IsectCapacity(16 * case["n"])
        while True:                     # sized once, from the first picture
            with torch.no_grad():
                _render(state, cap)
            try:
                cap.check()
                break
            except RuntimeError:
                continue
        state["capacity"] = cap
    return state


def _render(state, capacity):
    case = state["case"]
    return jaxsplat_amd.render(*state["params"], background=state["background"], block_size=case["block"],
                               adjoint=case["adjoint"], antialiased=case["antialiased"],
                               isect_capacity=capacity, **state["camera"])


def run(state):
    case, params = state["case"], state["params"]
    if case["call"] == "view":
        with torch.no_grad():
            return {"image": _render(state, None)}
    out = {}
    if case["call"] == "batch":
        image = state["renderer"](*params, state["viewmats"], state["backgrounds"], adjoint=case["adjoint"])
    elif case["call"] == "ops":
        cam = dict(state["camera"])
        viewmat = cam.pop("viewmat")
        xys, depths, radii, conics, hits, cum = jaxsplat_amd.project(
            *params[:3], viewmat, block_width=case["block"], adjoint=case["adjoint"], **cam)
        image = jaxsplat_amd.rasterize(params[3], params[4], state["background"], xys, depths, radii, conics, cum,
                                       img_shape=cam["img_shape"], block_width=case["block"],
                                       adjoint=case["adjoint"])
        out.update(xys=xys, conics=conics, depths=depths, radii=radii, hits=hits, cum=cum)
    else:
        image = _render(state, state["capacity"])
    out["image"] = image
    out["grads"] = dict(zip(_PARAMS, torch.autograd.grad(image, params, state["v_img"])))
    return out


def _blends(case):
    """About how many Gaussians a pixel blends, and how many a tile's list holds, from the sizes alone."""
    alpha = 0.75 if case["logit"] >= 2 else 0.3
    if case["scene"] == "random":
        cover = case["n"] * 0.04 / 36.0 * 64.0 / 16.0
    elif case["scene"] == "orbit":
        cover = case["n"] * 12.0 * math.exp(2 * case["log_scale"]) / 16.0
    else:
        width = 2.0 * 6.0 / 0.78 / 2.0      # the view's width at the middle of the depth range
        cover = case["n"] * 12.0 * math.exp(2 * case["log_scale"]) / (width * width * case["h"] / case["w"])
    return min(cover, 9.2 / alpha)


def work(case):
    gaussians, pixels = case["n"] * case["scenes"], case["h"] * case["w"] * case["views"]
    ch = case["channels"]
    backward = case["call"] != "view"
    row = 4 * (3 + 3 + 4 + ch + 1)          # a Gaussian's parameters, and its gradients
    bytes_ = gaussians * row * (2 if backward else 1) + pixels * 4 * ch * (2 if backward else 1)
    if case["call"] == "ops":
        bytes_ += gaussians * 4 * (2 + 3 + 1 + 1 + 1 + 1)
    # per blended (Gaussian, pixel) pair: the exponent and alpha 12, the blend 2 a channel; their adjoints twice that
    pair = (12 + 2 * ch) * (3 if backward else 1)
    # per projected (Gaussian, view): covariance, its projection and inverse, about 250; the adjoint twice that
    flops = pixels * _blends(case) * pair + gaussians * case["views"] / case["scenes"] * 250 * (3 if backward else 1)
    return {"bytes": bytes_, "flops": flops}


# -- the same in 64 bits --------------------------------------------------------

def _project64(means, scales, quats, vm, case, f, c):
    """xys, depths, conics, compensation, and the tile rectangles (x0, x1, y0, y1; empty where culled)."""
    h, w, bw = case["h"], case["w"], case["block"]
    tiles_x, tiles_y = -(-w // bw), -(-h // bw)
    rot, tr = vm[:3, :3], vm[:3, 3]
    t = means @ rot.T + tr
    x, y, z = t.unbind(1)
    seen = z.detach() > _CLIP
    z = torch.where(seen, z, torch.ones_like(z))
    qw, qx, qy, qz = quats.unbind(1)
    r = torch.stack([1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qw * qz), 2 * (qx * qz + qw * qy),
                     2 * (qx * qy + qw * qz), 1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qw * qx),
                     2 * (qx * qz - qw * qy), 2 * (qy * qz + qw * qx), 1 - 2 * (qx * qx + qy * qy)], 1).view(-1, 3, 3)
    m = r * scales[:, None, :]
    cov3 = m @ m.transpose(1, 2).contiguous()

    def cov2(tx, ty):
        zero = torch.zeros_like(z)
        j = torch.stack([f[0] / z, zero, -f[0] * tx / z ** 2, zero, f[1] / z, -f[1] * ty / z ** 2], 1).view(-1, 2, 3)
        a = j @ rot
        return a @ cov3 @ a.transpose(1, 2).contiguous()

    lx, ly = 1.3 * 0.5 * w / f[0], 1.3 * 0.5 * h / f[1]
    clamped = cov2(z * (x / z).clamp(-lx, lx), z * (y / z).clamp(-ly, ly))
    if case["adjoint"] == "reference":     # the reference differentiates at the mean that is not clamped
        free = cov2(x, y)
        clamped = free + (clamped - free).detach()
    a0, b, c0 = clamped[:, 0, 0], clamped[:, 0, 1], clamped[:, 1, 1]
    a, cc = a0 + 0.3, c0 + 0.3
    det = a * cc - b * b
    comp = ((a0 * c0 - b * b) / det).clamp(min=0).sqrt()
    conics = torch.stack([cc / det, -b / det, a / det], 1)
    xys = torch.stack([f[0] * x / (z + 1e-6) + c[0], f[1] * y / (z + 1e-6) + c[1]], 1)
    with torch.no_grad():
        half = 0.5 * (a + cc)
        radius = (3 * (half + (half * half - det).clamp(min=0.1).sqrt()).sqrt()).ceil()
        lo, hi = (xys - radius[:, None]) / bw, (xys + radius[:, None]) / bw + 1
        x0, x1 = (v.trunc().clamp(0, tiles_x).long() for v in (lo[:, 0], hi[:, 0]))
        y0, y1 = (v.trunc().clamp(0, tiles_y).long() for v in (lo[:, 1], hi[:, 1]))
        seen = seen & ((x1 - x0) * (y1 - y0) > 0)
        x1, y1 = torch.where(seen, x1, x0), torch.where(seen, y1, y0)
    return xys, z, conics, comp, seen, (x0, x1, y0, y1)


def _lists64(depths, rect, tiles_x, tiles):
    """The tiles' Gaussians from front to back, end to end, and where each tile's begin (tiles + 1)."""
    x0, x1, y0, y1 = rect
    order = torch.argsort(depths, stable=True)
    rank = torch.empty_like(order)
    rank[order] = torch.arange(order.numel(), device=order.device)
    count = (x1 - x0) * (y1 - y0)
    ids = torch.repeat_interleave(torch.arange(count.numel(), device=count.device), count)
    k = torch.arange(ids.numel(), device=ids.device) - (count.cumsum(0) - count)[ids]
    width = (x1 - x0)[ids]
    tile = (y0[ids] + k // width) * tiles_x + x0[ids] + k % width
    key, _ = torch.sort(tile * count.numel() + rank[ids])
    tile = key // count.numel()
    starts = torch.searchsorted(tile, torch.arange(tiles + 1, device=tile.device))
    return order[key - tile * count.numel()], starts


def _blend64(case, lists, starts, xys, conics, colors, opac, bg, v_img):
    """The image and, for a cotangent, the gradients of xys, conics, colors and opac."""
    h, w, bw, ch = case["h"], case["w"], case["block"], case["channels"]
    dev, tiles_x = xys.device, -(-w // bw)
    clamp = 0.99 if case["adjoint"] == "reference" else 0.999
    depth, per = 32, bw * bw
    image = torch.zeros((h * w, ch), dtype=torch.float64, device=dev)
    grads = None if v_img is None else [torch.zeros_like(t) for t in (xys, conics, colors, opac)]
    length = starts[1:] - starts[:-1]
    by_length = torch.argsort(length, descending=True)
    local = torch.arange(per, device=dev)
    for group in torch.split(by_length, max(1, (1 << 23) // (depth * per))):
        i = (group // tiles_x * bw)[:, None] + local // bw
        j = (group % tiles_x * bw)[:, None] + local % bw
        inside = (i < h) & (j < w)
        at = torch.where(inside, i * w + j, 0)
        px, py = j + 0.5, i + 0.5
        first, n = starts[group], length[group]

        def pairs(k0):
            k = k0 + torch.arange(depth, device=dev)
            here = k[None, :] < n[:, None]
            g = lists[torch.where(here, first[:, None] + k, 0)] if lists.numel() else torch.zeros_like(here).long()
            xy, cn = xys[g], conics[g]
            dx = xy[:, None, :, 0] - px[:, :, None]
            dy = xy[:, None, :, 1] - py[:, :, None]
            sigma = 0.5 * (cn[:, None, :, 0] * dx * dx + cn[:, None, :, 2] * dy * dy) + cn[:, None, :, 1] * dx * dy
            raw = opac[g][:, None, :, 0] * torch.exp(-sigma)
            ok = here[:, None, :] & (sigma >= 0) & (raw >= 1.0 / 255.0)
            return g, dx, dy, raw, ok

        t = torch.ones(px.shape, dtype=torch.float64, device=dev)
        done = ~inside
        total = torch.zeros((*px.shape, ch), dtype=torch.float64, device=dev)
        stops = []                      # per block: the entry within it that a pixel stops at
        for k0 in range(0, int(n[0]), depth):
            if bool(done.all()):
                break
            g, dx, dy, raw, ok = pairs(k0)
            alpha = torch.where(ok, raw.clamp(max=0.999), 0.0)
            after = t[:, :, None] * torch.cumprod(1 - alpha, 2)
            stop = ok & (after <= 1e-4)
            at_stop = torch.where(stop.any(2), stop.to(torch.uint8).argmax(2), depth)
            at_stop = torch.where(done, 0, at_stop)
            blends = torch.arange(depth, device=dev) < at_stop[:, :, None]
            alpha = torch.where(blends, alpha, 0.0)
            after = t[:, :, None] * torch.cumprod(1 - alpha, 2)
            before = torch.cat([t[:, :, None], after[:, :, :-1]], 2)
            total += (alpha * before) @ colors[g]
            t = after[:, :, -1]
            done = done | (at_stop < depth)
            stops.append(at_stop)
        image[at[inside]] = (total + t[:, :, None] * bg)[inside]
        if v_img is None:
            continue
        v = torch.where(inside[:, :, None], v_img.view(h * w, ch)[at], 0.0)
        behind = (t[:, :, None] * bg * v).sum(2)        # what is behind the entry, dotted with the cotangent
        for b in range(len(stops) - 1, -1, -1):
            g, dx, dy, raw, ok = pairs(b * depth)
            ok &= torch.arange(depth, device=dev) < stops[b][:, :, None]
            alpha = torch.where(ok, raw.clamp(max=clamp), 0.0)
            front = t[:, :, None] / torch.cumprod((1 - alpha).flip(2), 2).flip(2)
            cv = v @ colors[g].transpose(1, 2).contiguous()
            part = alpha * front * cv
            suffix = part.flip(2).cumsum(2).flip(2)
            v_alpha = torch.where(ok, front * cv - (suffix - part + behind[:, :, None]) / (1 - alpha), 0.0)
            if case["adjoint"] != "reference":
                v_alpha = torch.where(raw < clamp, v_alpha, 0.0)
            behind = behind + suffix[:, :, 0]
            t = front[:, :, 0]
            vs = -raw * v_alpha
            sums = torch.stack([vs.sum(1), (vs * dx).sum(1), (vs * dy).sum(1), (vs * dx * dx).sum(1),
                                (vs * dx * dy).sum(1), (vs * dy * dy).sum(1)], 2).view(-1, 6)
            g = g.reshape(-1)
            cn, o = conics[g], opac[g]
            grads[0].index_add_(0, g, torch.stack([cn[:, 0] * sums[:, 1] + cn[:, 1] * sums[:, 2],
                                                   cn[:, 1] * sums[:, 1] + cn[:, 2] * sums[:, 2]], 1))
            grads[1].index_add_(0, g, torch.stack([0.5 * sums[:, 3], sums[:, 4], 0.5 * sums[:, 5]], 1))
            grads[2].index_add_(0, g, ((alpha * front).transpose(1, 2).contiguous() @ v).reshape(-1, ch))
            grads[3].index_add_(0, g, -sums[:, :1] / o.clamp(min=1e-30))
    return image.view(h, w, ch), grads


def exact(case, seed):
    # deeper lists than the listed cases have would take too long in 64 bits
    if case["scene"] == "volume" and case["n"] * math.exp(2 * case["log_scale"]) > 10000:
        return None
    params, viewmats, backgrounds, f, c, v_img = _inputs(case, seed)
    p64 = [p.double() for p in params]
    vms, bgs = viewmats.double(), backgrounds.double()
    backward = case["call"] != "view"
    v64 = v_img.double().view(case["views"], case["h"], case["w"], -1) if backward else None
    tiles_x, tiles_y = -(-case["w"] // case["block"]), -(-case["h"] // case["block"])
    images, grads, out = [], [torch.zeros_like(p) for p in p64], {}
    for v in range(case["views"]):
        first = _view_scene(case, v) * case["n"]
        rows = slice(first, first + case["n"])
        leaf = [p[rows].clone().requires_grad_(backward) for p in p64]
        xys, depths, conics, comp, seen, rect = _project64(*leaf[:3], vms[v], case, f, c)
        opac = leaf[4] * comp[:, None] if case["antialiased"] else leaf[4]
        with torch.no_grad():
            lists, starts = _lists64(depths, rect, tiles_x, tiles_x * tiles_y)
            image, g = _blend64(case, lists, starts, xys, conics, leaf[3], opac, bgs[v], v64[v] if backward else None)
        images.append(image.reshape(-1, case["channels"]) if case["call"] == "batch" else image)
        if backward:
            through = torch.autograd.grad([xys, conics, opac], [leaf[0], leaf[1], leaf[2], leaf[4]],
                                          [g[0], g[1], g[3]])
            for k, d in zip((0, 1, 2, 4), through):
                grads[k][rows] += d
            grads[3][rows] += g[2]
        if case["call"] == "ops":
            on = seen.double()[:, None]
            out.update(xys=(xys * on).detach(), conics=None, depths=(depths[:, None] * on).detach(),
                       radii=None, hits=None, cum=None)
    out["image"] = torch.cat(images) if case["call"] == "batch" else images[0]
    if backward:
        out["grads"] = dict(zip(_PARAMS, grads))
    return out
