"""The tiles of the conv patch ordering, on the host: every layer that is accepted has a tile, within the kernel's limits
(a region of 8192 inputs, 159 KB of LDS), whatever its kernel, channels and alignment."""
import ctypes

import numpy as np
import pytest

from snntc_amd import _lib


def _tile(B, H, W, C, Kh, Kw, Sh=1, Sw=1, aligned=1):
    p = np.array([1e5, 0, 0, 1e-10, 1, 0, Kh, Kw, Sh, Sw, 1, 1.0], np.float32)
    t = (ctypes.c_int64 * 4)()
    rc = _lib.load().snntc_debug_order_tile(B, H, W, C, p.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), aligned, t)
    return rc, list(t)


# 14 patches each way for the smaller kernels, one patch for all of them; the channels run to the longest patch of 8192
@pytest.mark.parametrize("aligned", [1, 0])
@pytest.mark.parametrize("Kh", range(1, 33))
def test_every_layer_has_a_tile(Kh, aligned):
    for Kw in range(1, 33):
        longest = 8192 // (Kh * Kw)
        channels = range(1, longest + 1) if longest <= 300 else sorted(
            {*range(1, 300, 7), *range(4, longest + 1, 4 * max(1, longest // 400)), longest // 4 * 4, longest})
        for C in channels:
            H, W = (Kh + 13, Kw + 13) if Kh * Kw <= 9 else (Kh, Kw)
            rc, (th, tw, pixels, lds) = _tile(1, H, W, C, Kh, Kw, aligned=aligned)
            assert rc == _lib.OK, (Kh, Kw, C)
            P = Kh * Kw * C
            assert (th > 0) == (Kh * Kw > 1 and P > 128), (Kh, Kw, C)
            if th:
                region = (th - 1 + Kh) * (tw - 1 + Kw)
                assert region * C <= 8192 and 0 < lds <= 159 * 1024 and pixels in (0, region), (Kh, Kw, C)


def test_patches_beyond_the_limit_are_sorted():
    assert _tile(2, 20, 20, 33, 16, 16)[1] == [0, 0, 0, 0]          # 8448 inputs
    assert _tile(2, 20, 20, 16, 1, 1)[1] == [0, 0, 0, 0]            # nothing shared
