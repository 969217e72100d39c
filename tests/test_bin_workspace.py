"""Workspace sizes of the binning: jaxsplat_bin_emit_workspace_size serves a call
whatever number of intersections it expects, and the size for the number itself is
never larger.  No GPU calls."""

import ctypes

import pytest

from jaxsplat_amd import _lib


@pytest.mark.parametrize("n", [1, 2000, 12288, 70_000, 1_000_000])
@pytest.mark.parametrize("img", [(256, 256), (272, 272), (60, 4000), (1080, 1920), (5000, 400)],
                         ids=str)
def test_general_size_covers_every_expectation(n, img):
    L = _lib.lib()
    d = ctypes.byref(_lib.make_descriptor(n, img, (500.0, 500.0), (100.0, 100.0), 1.0, 0.01, 16))
    for cap in (1, 399_999, 1_000_001, 4_000_000, 100_000_000):
        size = L.jaxsplat_bin_emit_workspace_size(d, cap)
        each = [L.jaxsplat_bin_emit_workspace_size_expecting(d, cap, e)
                for e in (0, 1, 16 * n, 16 * n + 1, 1_000_001, 2_500_001, cap, 2 * cap)]
        assert size == max(each) and min(each) > 0
