"""The dense and patch gradients in each of their forms -- one, four, eight or sixteen wavefronts per tile of dX, four or eight
per tile of dW, with and without slices -- at ragged edges of tiles, chunks and pieces, against the fp64 oracle sums."""
import numpy as np
import pytest
import torch

from oracle import capi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


@pytest.mark.parametrize("B,I,J", [
    (1, 1, 17), (17, 33, 18), (15, 31, 63), (16, 32, 64), (17, 65, 65),   # one wavefront per tile, four; less and more than a tile
    (33, 40, 255), (20, 63, 257),                                         # eight and sixteen wavefronts
    (260, 520, 130), (700, 500, 40), (1100, 1000, 101),                   # many tiles: eight, one, four
    (129, 64, 300), (515, 127, 64), (1030, 300, 257),                     # slices of the samples
    (300, 1500, 1299), (512, 1300, 900),                                  # many tiles in one launch, and in parts: four wavefronts per tile of dW
    (2200, 63, 33), (4200, 64, 65),                                       # one and four tiles: more slices than sixteen
])
def test_dense_gradients(B, I, J):
    import snntc_amd as snn
    rng = np.random.default_rng(B + I + J)
    x = np.exp(rng.random((B, I))).astype(np.float32)
    x[rng.random((B, I)) < 0.1] = 1e5
    y = np.exp(1.2 * rng.random((B, J))).astype(np.float32)
    y[rng.random((B, J)) < 0.1] = 1e5
    x[0, : min(I, J)] = y[0, : min(I, J)]                                 # equal times count
    w = rng.standard_normal((I + 1, J)).astype(np.float32)
    out = np.concatenate([y, rng.random((B, J)).astype(np.float32)])
    g = np.zeros((2 * B, J), np.float32)
    g[:B] = rng.standard_normal((B, J))
    p = capi.fc_params(1.0)
    dx, dw, _ = (v.cpu().numpy() for v in snn.snnfc_grad(t(g), t(x), t(w), p, t(out)))
    again = snn.snnfc_grad(t(g), t(x), t(w), p, t(out))
    assert np.array_equal(dx, again[0].cpu().numpy()) and np.array_equal(dw, again[1].cpu().numpy())
    rdx, rdw, _ = capi.fc_backward_dev(g, x, w, p, out, wide=True)
    adx, adw, _ = capi.fc_backward_dev(np.abs(g), x, np.abs(w), p, out, wide=True)      # sums of absolute terms
    assert np.all(np.abs(dx - rdx) <= 1e-6 * np.abs(adx) + 1e-30)
    assert np.all(np.abs(dw - rdw) <= 1e-6 * np.abs(adw) + 1e-30)


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("B,I,J", [
    (1, 1, 128), (16, 32, 128), (17, 33, 129), (15, 64, 191), (33, 63, 320),                  # less than a tile, one, a bit more
    (63, 191, 1000), (208, 2000, 130), (240, 2000, 130),                                    # tiles of a turn of the chip, and of more
])
def test_dense_gradients_in_one_launch(B, I, J, bias):
    """dX and dW together, dW alone and dX alone: the same bits, and within the band of the fp64 sums."""
    import snntc_amd as snn
    rng = np.random.default_rng(B + I + J)
    x = np.exp(rng.random((B, I))).astype(np.float32)
    x[rng.random((B, I)) < 0.1] = 1e5
    y = np.exp(1.2 * rng.random((B, J))).astype(np.float32)
    y[rng.random((B, J)) < 0.1] = 1e5
    rcp = np.where(y < 1e5, rng.standard_normal((B, J)), np.inf).astype(np.float32)          # outputs that take no part weigh nothing
    w = rng.standard_normal((I + int(bias), J)).astype(np.float32)
    out = np.concatenate([y, rcp])
    g = np.zeros((2 * B, J), np.float32)
    g[:B] = rng.standard_normal((B, J))
    p = capi.fc_params(1.0 if bias else 0.0)
    args = (t(g), t(x), t(w), p, t(out))
    dx, dw, dp = snn.snnfc_grad(*args)
    assert not torch.any(torch.as_tensor(dp))
    assert torch.equal(dw, snn.snnfc_grad(*args, want_dx=False)[1])
    assert torch.equal(dx, snn.snnfc_grad(*args, want_dw=False)[0])
    dx, dw = dx.cpu().numpy(), dw.cpu().numpy()
    out[B:][y >= 1e5] = 0.0
    rdx, rdw, _ = capi.fc_backward_dev(g, x, w, p, out, wide=True)
    out[B:] = np.abs(out[B:])
    adx, adw, _ = capi.fc_backward_dev(np.abs(g), x, np.abs(w), p, out, wide=True)
    assert np.all(np.abs(dx - rdx) <= 1e-6 * np.abs(adx) + 1e-30)
    assert np.all(np.abs(dw - rdw) <= 1e-6 * np.abs(adw) + 1e-30)


@pytest.mark.parametrize("B,I,J", [
    (1, 1, 17), (129, 255, 17), (33, 64, 63), (40, 65, 64), (17, 31, 127),                    # dX tiles of one wavefront, of eight
    (352, 70, 130), (353, 70, 130), (448, 40, 50), (449, 40, 50),                             # slices, and few tiles
    (128, 200, 100), (240, 500, 50), (241, 500, 50), (240, 500, 33), (240, 447, 64), (240, 448, 64),   # eight tiles up to 240 rows and beyond, seven tiles
    (257, 300, 1000), (385, 511, 512), (412, 511, 512), (413, 511, 512), (448, 511, 512), (449, 511, 512), (448, 447, 512),    # 64 tiles up to 448 rows and beyond, 56
    (130, 100, 260), (131, 100, 260), (256, 784, 700), (300, 784, 770),                       # dX tiles first, dW tiles first
    (370, 2048, 1000), (430, 3000, 500), (446, 3300, 500), (100, 13000, 64), (100, 13100, 64),      # up to 3072 workgroups, and more
    (16, 8000, 1536), (16, 8000, 1559),                                                       # dW alone
])
def test_dense_gradients_whole_or_in_parts(B, I, J):
    """Both sides of the rules that choose one launch, the order of its tiles and their form, within the band of the fp64 sums."""
    import snntc_amd as snn
    rng = np.random.default_rng(B + I + J)
    x = np.exp(rng.random((B, I))).astype(np.float32)
    x[rng.random((B, I)) < 0.1] = 1e5
    y = np.exp(1.2 * rng.random((B, J))).astype(np.float32)
    y[rng.random((B, J)) < 0.1] = 1e5
    x[0, : min(I, J)] = y[0, : min(I, J)]
    w = rng.standard_normal((I + 1, J)).astype(np.float32)
    out = np.concatenate([y, rng.random((B, J)).astype(np.float32)])
    g = np.zeros((2 * B, J), np.float32)
    g[:B] = rng.standard_normal((B, J))
    p = capi.fc_params(1.0)
    args = (t(g), t(x), t(w), p, t(out))
    dx, dw, _ = snn.snnfc_grad(*args)
    alone = snn.snnfc_grad(*args, want_dx=False)[1].cpu().numpy()
    assert torch.equal(dx, snn.snnfc_grad(*args, want_dw=False)[0])                           # a sample's sums depend on J alone
    dx, dw = dx.cpu().numpy(), dw.cpu().numpy()
    rdx, rdw, _ = capi.fc_backward_dev(g, x, w, p, out, wide=True)
    adx, adw, _ = capi.fc_backward_dev(np.abs(g), x, np.abs(w), p, out, wide=True)
    # (a sum's partial sums of either sign stay well below its terms' absolute sum: a few roundings of that, as above)
    assert np.all(np.abs(dx - rdx) <= 1e-6 * np.abs(adx) + 1e-30)
    for got in (dw, alone):
        assert np.all(np.abs(got - rdw) <= 1e-6 * np.abs(adw) + 1e-30)


@pytest.mark.parametrize("B,I,J,slices", [(230, 300, 300, 13.55), (256, 512, 512, 12.88), (300, 128, 128, 12.04), (333, 512, 512, 11.69), (400, 500, 50, 10.89),
                                          (448, 200, 100, 10.17), (448, 300, 700, 10.30)])
def test_dense_weight_gradients_are_as_exact_in_one_launch(B, I, J, slices):
    """Samples that would be cut into slices (of 64 or more) are not summed in longer chains where one launch takes them."""
    import snntc_amd as snn
    rng = np.random.default_rng(B + I + J)
    x = np.exp(1.0 - rng.random((B, I))).astype(np.float32)
    y = np.exp(1.2 * rng.random((B, J))).astype(np.float32)
    w = rng.standard_normal((I + 1, J)).astype(np.float32)
    out = np.concatenate([y, rng.random((B, J)).astype(np.float32)])
    g = np.zeros((2 * B, J), np.float32)
    g[:B] = rng.standard_normal((B, J))
    p = capi.fc_params(1.0)
    dw = snn.snnfc_grad(t(g), t(x), t(w), p, t(out))[1].cpu().numpy()
    rdw, adw = (capi.fc_backward_dev(q, x, w, p, out, wide=True)[1] for q in (g, np.abs(g)))
    # `slices`: what the sum of slices of 64 samples and more shows on these inputs, in 1e-9 of the terms' absolute sum (the rounding of the
    # reference's results among it); one chain of additions per wavefront shows 13.0 to 14.7.  The margin is for another order of additions.
    error = (dw.astype(np.float64) - rdw)[adw != 0] / adw[adw != 0]
    assert np.sqrt(np.mean(error ** 2)) <= 1.03e-9 * slices


@pytest.mark.parametrize("B,H,W,C,Kc,S", [
    (2, 5, 9, 64, 64, 1), (2, 4, 10, 64, 128, 1), (1, 3, 11, 65, 16, 1), (1, 5, 16, 32, 64, 1), (2, 3, 18, 20, 32, 1),      # tiles of 8 to 128 pixels
    (1, 4, 19, 3, 64, 1), (1, 3, 30, 7, 48, 1), (2, 3, 31, 64, 80, 2), (1, 7, 34, 33, 64, 1), (3, 9, 8, 64, 256, 1), (1, 3, 3, 4, 16, 1),
    # strides that leave out slots: tiles of 8 pixels, of 16 to 128 with even strides, and odd strides that leave out none there
    (2, 7, 21, 64, 64, 2), (1, 5, 34, 64, 128, 2), (1, 7, 30, 64, 64, 3), (1, 9, 28, 65, 16, 4), (1, 6, 23, 128, 256, 5),
    (2, 6, 25, 32, 64, 2), (1, 5, 40, 16, 32, 2), (2, 4, 33, 7, 48, 2), (1, 6, 140, 3, 64, 2), (1, 5, 39, 16, 64, 4), (1, 7, 37, 30, 32, 6),
    (2, 5, 37, 32, 64, 3), (1, 4, 44, 9, 16, 3),
])
def test_conv_input_gradients_at_the_edges_of_tiles(B, H, W, C, Kc, S):
    """Three-column kernels: rows that begin or end with a padded column, or have none, in one image; the whole gradient and windows of it."""
    import snntc_amd as snn
    from snntc_amd import ops
    rng = np.random.default_rng(B + H + W + C + Kc)
    xpad = np.exp(rng.random((B, H, W, C))).astype(np.float32)
    xpad[rng.random(xpad.shape) < 0.1] = 1e5
    first, last = rng.random((B, H)) < 0.5, rng.random((B, H)) < 0.5
    xpad[:, :, 0][first] = 1e5
    xpad[:, :, -1][last] = 1e5
    p = capi.cv_params(3, 3, S, S, same=True, biasvolt=1.0)
    Nh, Nw, _ = capi.cv_dims(xpad.shape, p)
    w = rng.standard_normal((9 * C + 1, Kc)).astype(np.float32)
    out = np.concatenate([np.exp(1.2 * rng.random((B, Nh, Nw, Kc))), rng.standard_normal((B, Nh, Nw, Kc))]).astype(np.float32)
    dead = rng.random((B, Nh, Nw, Kc)) < 0.1
    out[:B][dead] = 1e5
    out[B:][dead] = 0.0
    g = np.zeros((2 * B, Nh, Nw, Kc), np.float32)
    g[:B] = rng.standard_normal((B, Nh, Nw, Kc))
    dx = snn.snncv_grad(t(g), t(xpad), t(w), p, t(out))[0].cpu().numpy()
    rdx, _, _ = capi.cv_backward_dev(g, xpad, w, p, out, wide=True)
    ao = out.copy()
    ao[B:] = np.abs(ao[B:])
    adx, _, _ = capi.cv_backward_dev(np.abs(g), xpad, np.abs(w), p, ao, wide=True)
    # (up to 2304 terms of either sign: partial sums stay near their square root, so the error stays near one rounding of |terms|)
    assert np.all(np.abs(dx - rdx) <= 2e-6 * np.abs(adx) + 1e-30)
    for h, wd, top, left in [(H - 2, W - 2, 1, 1), (1, W // 2 + 1, H // 2, 1), (H, W - 1, 0, 0), (2, 2, 0, W - 2)]:
        part = ops.snncv_grad(t(g), t(xpad), t(w), p, t(out), crop=(h, wd, top, left))[0].cpu().numpy()
        assert np.array_equal(part, dx[:, top:top + h, left:left + wd])


# Three-column kernels.  `slices`: what the form that the layer takes asks for, `least`: what a smaller workspace may come down to (the count of the
# blocks of 32 weight rows; where it is the larger one the workspace has room for it).  A layer that changes its form changes these.
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("B,H,W,C,Kc,Kh,Sh,slices,least", [
    # blocks of 32 rows
    (40, 8, 9, 32, 64, 3, 1, 26, 26), (9, 21, 23, 64, 65, 3, 1, 42, 42), (30, 12, 5, 64, 128, 3, 2, 7, 7), (60, 9, 4, 64, 64, 2, 1, 15, 15),
    (130, 6, 3, 96, 64, 3, 1, 8, 8), (7, 40, 12, 16, 40, 3, 1, 41, 41), (6, 22, 22, 80, 33, 1, 1, 32, 32),
    # sixteen channels a wavefront: rows of 17, 7, 1, 2 and 7 patches; 80 channels, two kernel rows
    (20, 9, 19, 48, 130, 3, 1, 18, 34), (25, 10, 9, 256, 65, 3, 1, 8, 7), (120, 21, 3, 256, 66, 3, 2, 8, 7), (60, 21, 4, 256, 66, 3, 2, 8, 7),
    (40, 8, 9, 256, 70, 3, 1, 8, 7), (30, 12, 12, 80, 70, 2, 1, 25, 48),
])
def test_conv_weight_gradients_by_pixels(B, H, W, C, Kc, Kh, Sh, slices, least, bias):
    """Runs of patches that begin and end within rows and images, the last slices without a patch for some wavefronts."""
    _check_weight_gradients(B, H, W, C, Kc, Kh, Sh, slices, least, bias)


@pytest.mark.parametrize("B,H,W,C,Kc,Kh,Sh,slices,least,bias", [
    (75, 10, 9, 256, 65, 3, 1, 16, 7, True), (205, 21, 3, 512, 65, 3, 2, 8, 6, True), (103, 21, 4, 512, 65, 3, 2, 8, 6, False), (192, 9, 4, 512, 65, 2, 1, 12, 8, True),
    (60, 30, 30, 64, 33, 2, 1, 192, 128, False),
])
def test_conv_weight_gradients_by_pixels_of_32_channels(B, H, W, C, Kc, Kh, Sh, slices, least, bias):
    """The launches that fill the chip: rows of 7, 1, 2, 2 and 28 patches, row strides of two, two kernel rows, outputs that are no multiple of 64."""
    _check_weight_gradients(B, H, W, C, Kc, Kh, Sh, slices, least, bias, _weight_gradients_64)


def _weight_gradients_oracle(g, x, w, p, out):
    """dW and the sums of its terms' sizes."""
    sizes = out.copy()
    sizes[len(x):] = np.abs(sizes[len(x):])
    return capi.cv_backward_dev(g, x, w, p, out, wide=True)[1], np.abs(capi.cv_backward_dev(np.abs(g), x, w, p, sizes, wide=True)[1])


def _weight_gradients_64(g, x, w, p, out):
    """The same in plain 64-bit arithmetic on the GPU, tap by tap (hundreds of millions of terms)."""
    B, _, _, C = x.shape
    Nh, Nw, Kc = out.shape[1:]
    Kh, Sh, biasvolt = int(p[6]), int(p[8]), float(p[11])
    upstream = (t(g[:B]).double() * t(out[B:]).double()).reshape(-1, Kc)
    times = t(out[:B]).double().reshape(-1, Kc)
    xd = t(x).double()
    sums, sizes = (torch.zeros(w.shape, dtype=torch.float64, device=DEV) for _ in range(2))
    taps = [xd[:, kh:kh + (Nh - 1) * Sh + 1:Sh, kw:kw + Nw].reshape(-1, C) for kh in range(Kh) for kw in range(3)]
    if len(w) > 3 * Kh * C:
        taps.append(torch.full((B * Nh * Nw, 1), biasvolt, dtype=torch.float64, device=DEV))
    for tap, inputs in enumerate(taps):
        rows = slice(tap * C, tap * C + inputs.shape[1])
        for s in range(0, len(inputs), 512):
            terms = (inputs[s:s + 512, :, None] - times[s:s + 512, None]).clamp(max=0) * upstream[s:s + 512, None]
            sums[rows] += terms.sum(0)
            sizes[rows] += terms.abs().sum(0)
    return sums.cpu().numpy(), sizes.cpu().numpy()


# (`blocks`: the error of the blocks of 32 weight rows on these inputs)
@pytest.mark.parametrize("B,H,W,C,Kc,blocks", [
    (32, 9, 9, 144, 100, 5.096), (16, 9, 9, 112, 128, 6.743), (7, 40, 12, 48, 40, 3.902), (15, 7, 25, 144, 96, 4.964), (18, 20, 7, 144, 48, 4.783),
    (11, 20, 14, 48, 100, 4.122), (65, 9, 9, 96, 100, 3.873), (4, 16, 16, 512, 512, 13.979),
])
def test_conv_weight_gradients_are_as_exact_by_pixels(B, H, W, C, Kc, blocks):
    """A wavefront that walks over pixels, eight to a workgroup, rounds no more than the blocks of 32 weight rows do."""
    assert _conv_weight_gradient_error(B, H, W, C, Kc) <= 1.005 * blocks


def _conv_weight_gradient_error(B, H, W, C, Kc):
    """rms error of dW, in 1e-9 of the terms' absolute sum."""
    import snntc_amd as snn
    rng = np.random.default_rng(B + H + W + C + Kc)
    x = np.exp(1.0 - rng.random((B, H, W, C))).astype(np.float32)
    p = capi.cv_params(3, 3, 1, 1, same=False, biasvolt=1.0)
    w = rng.standard_normal((9 * C + 1, Kc)).astype(np.float32)
    y = np.exp(1.2 * rng.random((B, H - 2, W - 2, Kc))).astype(np.float32)
    g = np.zeros((2 * B, H - 2, W - 2, Kc), np.float32)
    g[:B] = rng.standard_normal(y.shape)
    out = np.concatenate([y, np.ones_like(y)])                # (upstream values without a rounding of their own)
    dw = snn.snncv_grad(t(g), t(x), t(w), p, t(out))[1].cpu().numpy().astype(np.float64)
    rdw, adw = _weight_gradients_64(g, x, w, p, out)
    return 1e9 * np.sqrt(np.mean(((dw - rdw) / adw) ** 2))


def _check_weight_gradients(B, H, W, C, Kc, Kh, Sh, slices, least, bias, reference=_weight_gradients_oracle):
    import ctypes
    import snntc_amd as snn
    from snntc_amd import _lib
    rng = np.random.default_rng(B + H + W + C + Kc)
    x = np.exp(rng.random((B, H, W, C))).astype(np.float32)
    x[rng.random(x.shape) < 0.1] = 1e5
    p = capi.cv_params(Kh, 3, Sh, 1, same=False, biasvolt=1.0 if bias else 0.0)
    Nh, Nw, _ = capi.cv_dims(x.shape, p)
    w = rng.standard_normal((Kh * 3 * C + int(bias), Kc)).astype(np.float32)
    out = np.concatenate([np.exp(1.2 * rng.random((B, Nh, Nw, Kc))), rng.standard_normal((B, Nh, Nw, Kc))]).astype(np.float32)
    dead = rng.random((B, Nh, Nw, Kc)) < 0.1
    out[:B][dead] = 1e5
    out[B:][dead] = 0.0
    g = np.zeros((2 * B, Nh, Nw, Kc), np.float32)
    g[:B] = rng.standard_normal((B, Nh, Nw, Kc))
    dw = snn.snncv_grad(t(g), t(x), t(w), p, t(out))[1]
    rdw, adw = reference(g, x, w, p, out)
    # (some thousand terms of either sign, 2e-7 of |terms| as for the dense gradients' partial sums, and a margin)
    assert np.all(np.abs(dw.cpu().numpy() - rdw) <= 2e-6 * adw + 1e-30)
    # with the room that the kernels for any shape ask for there are fewer slices, and with less the call is refused
    lib = _lib.load()
    need = ctypes.c_size_t()
    fp = np.ascontiguousarray(p, np.float32).ctypes.data_as(ctypes.POINTER(ctypes.c_float))
    _lib.check(lib.snntc_cv_backward_workspace_bytes(B, H, W, C, Kc, fp, ctypes.byref(need)))
    args = [t(g), t(x), t(w), t(out)]
    again = torch.empty_like(dw)
    stream = torch.cuda.current_stream().cuda_stream
    ws = torch.empty(need.value, dtype=torch.uint8, device=DEV)
    ptr = lambda a: a.data_ptr() if a is not None else None                      # noqa: E731
    call = lambda n: lib.snntc_cv_backward(ptr(args[0]), ptr(args[1]), ptr(args[2]), fp, ptr(args[3]), None, ptr(again), None, B, H, W, C, Kc,   # noqa: E731
                                           w.shape[0], 2 * B, ptr(ws), n, stream)
    align = lambda floats: -(-4 * floats // 256) * 256                           # noqa: E731
    P, S = Kh * 3 * C, B * Nh * Nw
    others = align(S * Kc) + align((P + 1) * Kc) + (align(S * P) if Kc % 16 else 0)          # (the last for dX of such layers)
    partial = lambda n: others + (align(n * (P + 1) * Kc) if n > 1 else 0)                   # noqa: E731
    assert need.value == partial(max(slices, least))
    assert call(need.value) == _lib.OK
    assert torch.equal(again, dw)
    fewer = 0
    for room in range(need.value - 256, 0, -max(256, need.value // 40 // 256 * 256)):
        if call(room) != _lib.OK:
            break
        err = np.abs(again.cpu().numpy() - rdw)
        assert np.all(err <= 2e-6 * adw + 1e-30)
        fewer += 1
    else:
        raise AssertionError("no workspace was refused")
    assert (fewer > 0) == (slices > least)
    assert call(partial(least)) == _lib.OK and call(partial(least) - 256) != _lib.OK
