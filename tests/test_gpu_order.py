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


ROWS = [(1536, 257), (2560, 257), (8192, 260), (8193, 260), (1536, 512), (100, 513), (128, 784), (100, 1023), (101, 1024), (3, 1025), (2, 2048), (5, 2049), (3, 4096), (2, 4097), (2, 8191),
        (3, 8192)]


@pytest.mark.parametrize("kind", ["plain", "silent", "crowded", "signs", "repeats", "bytes", "ink", "one", "odd"])
@pytest.mark.parametrize("B,I", ROWS)
def test_dense_row_order(B, I, kind):
    """Dense rows that are ranked (or, where values repeat, sorted by a network after all), at the edges of their length classes."""
    import snntc_amd as snn
    rng = np.random.default_rng(B * 7 + I)
    if kind in ("ink", "one", "odd"):
        x = np.full((B, I), np.float32(np.e))
        if kind == "ink":                                   # mostly background, the rest in 256 levels
            ink = rng.random((B, I)) < 0.2
            x[ink] = np.exp(1.0 - rng.integers(1, 256, ink.sum()) / 255.0).astype(np.float32)
        elif kind == "odd":                                 # infinities, NaN of both signs, zeros of both, the smallest numbers
            x = np.exp(rng.random((B, I))).astype(np.float32)
            pick = np.array([np.inf, -np.inf, np.nan, -np.nan, 0.0, -0.0, 1e-45, -1e-45, 3.4e38, 1e5, 1e5 - 0.1], np.float32)
            some = rng.random((B, I)) < 0.2
            x[some] = pick[rng.integers(0, len(pick), some.sum())]
    else:
        x = _values(kind, rng, (B, 1, 1, I)).reshape(B, I)
    xt = torch.from_numpy(x).to(DEV)
    w = torch.from_numpy(rng.standard_normal((I + 1, 3)).astype(np.float32)).to(DEV)
    _, z, perm, _ = snn.snnfc(xt, w, capi.fc_params(1.0), return_aux=True)
    bits = np.where(x == 0, np.float32(0), x).view(np.uint32)
    key = np.where(bits >> 31 == 1, ~bits, bits | np.uint32(0x80000000))
    want = np.argsort(key, axis=1, kind="stable")
    assert np.array_equal(perm.cpu().numpy(), want)
    assert np.array_equal(z.cpu().numpy().view(np.uint32), np.take_along_axis(bits, want, 1))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("B,I", [(128, 784), (128, 785), (4, 3000)])
def test_dense_rows_at_any_alignment(B, I, offset):
    import snntc_amd as snn
    from oracle.capi import fc_forward_dev
    rng = np.random.default_rng(I + offset)
    x = np.exp(rng.random((B, I))).astype(np.float32)
    w = (4.0 / I + rng.standard_normal((I + 1, 40)) / np.sqrt(I)).astype(np.float32)
    room = torch.zeros(B * I + 1, device=DEV)
    view = room[offset:offset + B * I].view(B, I)
    view.copy_(torch.from_numpy(x))
    out = snn.snnfc(view, torch.from_numpy(w).to(DEV), capi.fc_params(1.0))
    ref = fc_forward_dev(x, w, capi.fc_params(1.0))
    assert np.array_equal(out.cpu().numpy().view(np.uint32), (ref[0] if isinstance(ref, tuple) else ref).view(np.uint32))


def _tied_rows(kind, rng, B, I):
    x = np.exp(rng.random((B, I))).astype(np.float32)
    if kind == "levels":                                    # every bucket a single value; a tenth silent, a row of one value
        x = np.exp(rng.integers(0, 200, (B, I)) / 200.0).astype(np.float32)
        x[rng.random((B, I)) < 0.1] = 1e5
        x[B // 2] = 1.5
    elif kind == "runs":                                    # the same in long runs of equal neighbours
        x = np.exp((np.arange(I) // 37 * 11 % 50 + rng.integers(0, 3, (B, 1))) / 60.0).astype(np.float32)
    elif kind in ("lowest", "middle", "highest"):           # one value in two inputs, the others different, on both sides or one
        x[rng.random((B, I)) < 0.5] = {"lowest": 0.5, "middle": 1.7, "highest": 3.0}[kind]
        x[:, ::41] = 1e5
        x[B // 2, : I // 2] = 1e5
    elif kind == "close":                                   # ... and next to it within its bucket
        x[rng.random((B, I)) < 0.5] = 1.7
        x[:, ::5] = (np.float32(1.7) + rng.integers(-9, 9, x[:, ::5].shape) * np.float32(2.0 ** -20)).astype(np.float32)
    elif kind == "two":                                     # two values among different ones: one of them stays in the bitmap
        x[rng.random((B, I)) < 0.4] = 1.7
        x[rng.random((B, I)) < 0.3] = 2.1
    elif kind == "octave":                                  # crowded, all different, with outliers
        x = (2 + 0.2 * rng.random((B, I))).astype(np.float32)
        far = rng.random((B, I)) < 0.03
        x[far] = np.exp(rng.uniform(0, 11, int(far.sum())))
    elif kind == "zeros":
        x = np.where(rng.random((B, I)) < 0.6, rng.choice(np.array([0.0, -0.0], np.float32), (B, I)), rng.standard_normal((B, I))).astype(np.float32)
    return x


TIED_ROWS = [(2048, 260), (6144, 512), (3072, 449), (300, 513), (1024, 784), (300, 1023), (400, 1024),     # edges of the rule and of the forms
             (1, 1025), (256, 1028), (257, 1025), (3, 2047), (256, 2048), (257, 2048), (2, 2049), (3, 4096), (2, 4097), (3, 8192)]


@pytest.mark.parametrize("kind", ["levels", "runs", "lowest", "middle", "highest", "close", "two", "octave", "zeros"])
@pytest.mark.parametrize("B,I", TIED_ROWS)
def test_dense_rows_whose_values_repeat(B, I, kind):
    """Counted rows, rows with one value out of the bitmap, rows ranked as they are and rows that go to a network: order, causal sets, outputs."""
    import snntc_amd as snn
    rng = np.random.default_rng(B * 3 + I)
    x = _tied_rows(kind, rng, B, I)
    w = (4.0 / I + rng.standard_normal((I + 1, 3)) / np.sqrt(I)).astype(np.float32)
    p = capi.fc_params(1.0)
    ref_out, ref_k, ref_sorted, ref_perm = capi.fc_forward_dev(x, w, p, want_aux=True)
    out, sz, perm, ck = (v.cpu().numpy() for v in snn.snnfc(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV), p, return_aux=True))
    assert np.array_equal(perm, ref_perm)
    assert np.array_equal(sz, ref_sorted)
    assert np.array_equal(ck, ref_k)
    assert np.array_equal(out.view(np.uint32), ref_out.view(np.uint32))


def _odd_rows(rng, B, I):
    x = np.exp(rng.random((B, I))).astype(np.float32)
    pick = np.array([np.inf, -np.inf, np.nan, -np.nan, 0.0, -0.0, 1e-45, -1e-45, 3.4e38, 1e5, 1e5 - 0.1], np.float32)
    some = rng.random((B, I)) < 0.2
    some[: B // 2] &= rng.random((B // 2, 1)) < 0.5          # rows without any among them
    x[some] = pick[rng.integers(0, len(pick), some.sum())]
    return torch.from_numpy(x).to(DEV)


@pytest.mark.parametrize("I", [513, 784, 1024])
def test_odd_values_take_part_alike_in_ranked_and_sorted_rows(I):
    """Infinities and NaN of both signs: which inputs a scan walks (n_real) does not depend on how its row was ordered."""
    import snntc_amd as snn
    rng = np.random.default_rng(I)
    x = _odd_rows(rng, 600, I)
    w = torch.from_numpy((4.0 / I + rng.standard_normal((I + 1, 40)) / np.sqrt(I)).astype(np.float32)).to(DEV)
    p = capi.fc_params(1.0)
    out, z, perm, ck = snn.snnfc(x, w, p, return_aux=True)                               # ranked
    few, z2, perm2, ck2 = snn.snnfc(x[150:449].contiguous(), w, p, return_aux=True)      # a network
    assert torch.equal(perm[150:449], perm2) and torch.equal(ck[150:449], ck2)
    assert torch.equal(z[150:449].view(torch.int32), z2.view(torch.int32))
    assert torch.equal(out[150:449].view(torch.int32), few[:299].view(torch.int32))
    assert torch.equal(out[750:1049].view(torch.int32), few[299:].view(torch.int32))


@pytest.mark.parametrize("B,I,J", [(5, 784, 30), (3, 300, 16), (4, 1024, 100), (7, 129, 10)])
def test_odd_values_take_part_alike_where_the_scan_orders_its_rows(B, I, J):
    import snntc_amd as snn
    rng = np.random.default_rng(I)
    x = _odd_rows(rng, B, I)
    w = torch.from_numpy((4.0 / I + rng.standard_normal((I + 1, J)) / np.sqrt(I)).astype(np.float32)).to(DEV)
    p = capi.fc_params(1.0)
    own = snn.snnfc(x, w, p)                                # (asked for the order, a launch of its own makes it)
    assert torch.equal(own.view(torch.int32), snn.snnfc(x, w, p, return_aux=True)[0].view(torch.int32))
