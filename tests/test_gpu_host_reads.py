"""The host side of the fused render: counts read through a pinned word, and the
two buffers that its backward keeps.

All results must equal an undisturbed render's bit for bit: from several threads
and streams at once, behind more work than the reader polls for, with
saved-tensor hooks that hand back misaligned copies, and where the backward falls
back to the separate adjoints (those within the order of the float additions,
1e-5 |g| + 1e-6 max|g|).  A capturing stream refuses the read.
"""

import threading

import numpy as np
import pytest

from jaxsplat_amd import IsectCapacity, _ops, render, scenes
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _scene(seed, n=2500):
    rng = np.random.default_rng(seed)
    return [H.dev(a) for a in scenes.gaussians(rng, n, (-2, -1.5, 2), (2, 1.5, 6), np.log(0.05))]


def _step(params, size, capacity=None):
    t = H.torch()
    h, w = size
    p = [x.detach().requires_grad_(True) for x in params]
    img = render(*p, viewmat=H.dev(scenes.IDENTITY), background=t.full((3,), 0.25, device="cuda"),
                 img_shape=size, f=(float(w), float(w)), c=(w / 2, h / 2), glob_scale=1.0,
                 clip_thresh=0.01, isect_capacity=capacity)
    v = t.linspace(-1, 1, img.numel(), device="cuda").view(img.shape)
    return [img.detach()] + list(t.autograd.grad(img, p, v))


def _same(a, b):
    return all(np.array_equal(H.host(x).view(np.uint32), H.host(y).view(np.uint32))
               for x, y in zip(a, b))


SIZES = [(100, 90), (300, 260)]         # one radix pass of pairs; binned by rows


@pytest.mark.parametrize("size", SIZES, ids=str)
def test_threads_and_streams(size):
    t = H.torch()
    inputs = [_scene(s, 400 * (s + 1)) for s in range(4)]
    want = [_step(p, size) for p in inputs]
    t.cuda.synchronize()
    bad = []

    def work(i):
        try:
            with t.cuda.stream(t.cuda.Stream()):
                for _ in range(10):
                    if not _same(_step(inputs[i], size), want[i]):
                        bad.append(i)
        except Exception as e:          # reported by the main thread
            bad.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad


@pytest.mark.parametrize("size", SIZES, ids=str)
def test_behind_long_work_and_hooks(size):
    t = H.torch()
    p = _scene(1)
    want = _step(p, size)
    a = t.randn(8192, 8192, device="cuda")
    for _ in range(4):                  # tens of ms queued before the count
        a = (a @ a).clamp_(-1, 1)
    assert _same(_step(p, size), want)

    def pack(x):
        return x.dtype, x.shape, x.contiguous().view(-1)

    def unpack(s):
        dtype, shape, flat = s
        big = t.empty(flat.numel() + 1, dtype=dtype, device="cuda")
        big[1:] = flat
        return big[1:].view(shape)

    with t.autograd.graph.saved_tensors_hooks(pack, unpack):
        assert _same(_step(p, size), want)


@pytest.mark.parametrize("size", SIZES, ids=str)
def test_fallback_backward(size, monkeypatch):
    p = _scene(2)
    want = _step(p, size)
    monkeypatch.setattr(_ops, "STAGED_BACKWARD", False)
    got = _step(p, size)
    assert _same(got[:1], want[:1])
    for g, w in zip(got[1:], want[1:]):
        ref = H.host(w).astype(np.float64)
        assert np.all(np.abs(H.host(g) - ref) <= 1e-5 * np.abs(ref) + 1e-6 * np.abs(ref).max())


def test_capturing_stream_refuses_the_read():
    t = H.torch()
    p = _scene(3, 300)
    size = SIZES[0]
    cap = IsectCapacity(1 << 16)
    want = _step(p, size, cap)
    cap.check()
    side = t.cuda.Stream()
    side.wait_stream(t.cuda.current_stream())
    g = t.cuda.CUDAGraph()
    with pytest.raises(RuntimeError):
        with t.cuda.graph(g, stream=side):
            _step(p, size)
    t.cuda.synchronize()
    assert _same(_step(p, size, cap), want) and _same(_step(p, size), want)
    assert cap.check() > 0


@pytest.mark.parametrize("adjoint", ["reference", "consistent"])
@pytest.mark.parametrize("nch", [1, 3])
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_antialiased_fused_equals_composition(size, nch, adjoint, monkeypatch):
    """The antialiased render as one node: images and gradients bit for bit those
    of the projection, the product and the rasterization as separate nodes."""
    t = H.torch()
    h, w = size
    params = _scene(5)
    params[1] = params[1] * 0.2         # footprints below a pixel: compensation well below 1
    params[3] = params[3][:, :nch].contiguous()
    v = t.linspace(-1, 1, h * w * nch, device="cuda").view(h, w, nch)

    def step(staged=True):
        monkeypatch.setattr(_ops, "STAGED_BACKWARD", staged)
        p = [x.detach().requires_grad_(True) for x in params]
        img = render(*p, viewmat=H.dev(scenes.IDENTITY), background=v[0, 0].abs().contiguous(),
                     img_shape=size, f=(float(w), float(w)), c=(w / 2, h / 2), glob_scale=1.0,
                     clip_thresh=0.01, adjoint=adjoint, antialiased=True)
        return [img.detach()] + list(t.autograd.grad(img, p, v))

    fused, atomic = step(), step(staged=False)
    monkeypatch.setattr(_ops, "FUSED_RENDER", False)
    separate = step()
    assert _same(fused, separate)
    for g, s in zip(atomic, separate):
        ref = H.host(s).astype(np.float64)
        assert np.all(np.abs(H.host(g) - ref) <= 1e-5 * np.abs(ref) + 1e-6 * np.abs(ref).max())
