"""The conv patch ordering in each of its forms -- patches by a wavefront or by the workgroup, bitmaps from pixels or
from the patches' own inputs, aligned and single loads -- at the edges of its length classes and tiles, for values that
crowd, repeat, change sign or never spiked, against the oracle's stable order."""
import numpy as np
import pytest
import torch

from oracle import capi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

FORMS = [
    # B, H, W, C, Kh, Kw, Sh, Sw
    (8, 27, 31, 13, 5, 1, 1, 1),        # P = 65: the shortest (many patches), one iteration, single loads
    (2, 19, 17, 16, 3, 3, 1, 1),        # P = 144: bits set by the patches
    (2, 18, 35, 64, 1, 3, 1, 1),        # P = 192 and, below, 288: bits from pixels; ragged last tiles
    (2, 13, 21, 32, 3, 3, 1, 1),
    (3, 21, 23, 3, 7, 7, 2, 2),         # strided, row of 3 channels
    (2, 11, 12, 36, 3, 3, 1, 2),        # P = 324: the first of nine iterations
    (1, 17, 18, 64, 3, 3, 1, 1),        # P = 576, and 577 in one column
    (2, 9, 3, 577, 2, 1, 1, 1),
    (1, 9, 10, 128, 3, 3, 1, 1),        # P = 1152, the longest of a wavefront
    (2, 5, 6, 289, 2, 2, 2, 3),         # P = 1156: the workgroup's shortest; gaps between the patches
    (1, 7, 8, 256, 3, 3, 1, 1),
    (1, 5, 9, 160, 4, 4, 1, 1),         # P = 2560
    (1, 4, 5, 321, 4, 2, 1, 1),         # P = 2568
    (1, 6, 5, 512, 3, 3, 1, 1),
    (1, 3, 4, 2048, 2, 2, 1, 2),        # P = 8192, the longest
    (1, 8, 8, 164, 7, 7, 1, 1),         # P = 8036 and, below, 4896 (the shortest), 8192: no room for a bitmap per pixel
    (1, 10, 21, 32, 9, 17, 1, 2),
    (2, 16, 17, 32, 16, 16, 1, 1),
]


def _values(kind, rng, shape):
    x = np.exp(rng.random(shape)).astype(np.float32)
    if kind == "silent":                                    # a third never spiked, two of them at other late times; one image none
        x[rng.random(shape) < 0.33] = 1e5
        x[0, 0, 0, :2] = (2e5, 3e5)
        x[-1] = 1e5
    elif kind == "crowded":                                 # nearly all within 200 steps of one value, a few decades away
        x = (np.float32(1.5) + rng.integers(0, 200, shape) * np.float32(2.0 ** -23)).astype(np.float32)
        far = rng.random(shape) < 0.01
        x[far] = np.exp(rng.uniform(-9, 9, int(far.sum())))
    elif kind == "signs":                                   # both signs and both zeros
        x = rng.standard_normal(shape).astype(np.float32)
        x[rng.random(shape) < 0.01] = 0.0
        x[rng.random(shape) < 0.01] = -0.0
    elif kind == "bytes":                                   # an 8-bit image with a saturated part and one of a single value
        x = np.exp(1.0 - rng.integers(0, 256, shape) / 255.0).astype(np.float32)
        x[:, : shape[1] // 3] = 1.0
        x[-1] = 1.5
    elif kind == "repeats":                                 # half the inputs share one value
        x[rng.random(shape) < 0.5] = 1.25
    return x


@pytest.mark.parametrize("kind", ["plain", "silent", "crowded", "signs", "repeats", "bytes"])
@pytest.mark.parametrize("B,H,W,C,Kh,Kw,Sh,Sw", FORMS)
def test_patch_order(B, H, W, C, Kh, Kw, Sh, Sw, kind):
    import snntc_amd as snn
    rng = np.random.default_rng(H * W * C)
    x = _values(kind, rng, (B, H, W, C))
    w = (rng.standard_normal((Kh * Kw * C + 1, 4)) * 0.3 + 0.05).astype(np.float32)
    p = capi.cv_params(Kh, Kw, Sh, Sw, same=False)
    ref_out, ref_k, ref_sorted, ref_perm = capi.cv_forward_dev(x, w, p, want_aux=True)
    out, sz, perm, ck = (v.cpu().numpy() for v in snn.snncv(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV), p,
                                                            return_aux=True))
    assert np.array_equal(perm, ref_perm), "permutation differs"
    assert np.array_equal(sz, ref_sorted)
    assert np.array_equal(ck, ref_k)
    assert np.array_equal(out.view(np.uint32), ref_out.view(np.uint32))
