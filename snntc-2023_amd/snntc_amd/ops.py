"""The four SNN-TC ops over PyTorch-ROCm tensors, each a thin call into the C ABI.

Counterparts of the reference's op handles (SNN_TC_Modules.py:29-33, 89-93):

    snnfc(X, W, Params)                      -> Y[2B, J]
    snnfc_grad(grad, X, W, Params, Y)        -> (dX, dW, dParams)
    snncv(Xpad, W, Params)                   -> Y[2B, Nh, Nw, Kc]
    snncv_grad(grad, Xpad, W, Params, Y)     -> (dXpad, dW, dParams)

``SnnFc`` / ``SnnCv`` are the differentiable ops that replace ``@ops.RegisterGradient``.
Tensors must be float32 on a ROCm device; ``Params`` is the host-side float32 vector the layers
build.  PyTorch supplies device memory, the current HIP stream and the autograd engine; the host side
of a call (checks, allocation, launches, graph nodes) is csrc/binding.cpp.  The differentiable ops are
``torch.autograd.Function`` classes whose ``apply`` is that native path; it hands a call with forward-mode
tangents, functorch transforms, tracers or tensor wrappers in it to the function itself (``GENERAL``).
"""
import ctypes

import numpy as np
import torch

from . import _lib

_giveups_seen = {}


def check_scan_health(device=None):
    """Raises SnntcError if, since the last call for this device, a wavefront of the classifier-head scan
    ran out of its bounded wait (the affected outputs are NaN).  Synchronises with the current stream of
    the device: call it where the program waits for the GPU anyway (after reading a loss, at the end of
    an epoch or of a batch of requests)."""
    device = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    with torch.cuda.device(device):
        n = _lib.scan_giveups(torch.cuda.current_stream(device).cuda_stream)
    before = _giveups_seen.get(device.index, 0)
    _giveups_seen[device.index] = n
    if n > before:
        raise _lib.SnntcError(_lib.ERR_HIP, f"{n - before} scan wavefront(s) gave up waiting for partial sums on "
                                            f"{device}: the outputs of their work items are NaN")
    return n


def _params(params, n):
    p = _lib.params_array(params, n)
    return p, p.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


def _dev_f32(t, name, ndim):
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{name} must be a torch.Tensor")
    if not t.is_cuda:
        raise _lib.SnntcLibraryError(
            f"{name} lives on {t.device}: the SNN-TC ops run on a ROCm GPU only (no CPU fallback)")
    if t.dtype != torch.float32:
        raise TypeError(f"{name} must be float32, got {t.dtype}")
    if t.dim() != ndim:
        raise ValueError(f"{name} must have {ndim} dimensions, got shape {tuple(t.shape)}")
    return t.contiguous()


def release_workspaces():
    """Gives unused scratch memory back to the device.  The ops take their scratch from PyTorch's caching
    allocator call by call, so this drops what that allocator keeps."""
    if torch.cuda.is_initialized():
        torch.cuda.empty_cache()


def _stream(device):
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def snnfc(X, W, Params, return_aux=False):
    """Dense forward.  X[B,I], W[I+bias,J] -> Y[2B,J] (spike times ; 1/(sum w - theta)).
    With return_aux=True also returns (sorted_z[B,I], perm[B,I] int32, causal_k[B,J] int32)."""
    if not return_aux:
        return _lib.native().fc_forward(X, W, Params)
    lib = _lib.load()
    X = _dev_f32(X, "X", 2)
    W = _dev_f32(W, "W", 2)
    p, pp = _params(Params, 6)
    B, I = X.shape
    w_rows, J = W.shape
    with torch.cuda.device(X.device):
        need = ctypes.c_size_t()
        _lib.check(lib.snntc_fc_forward_workspace_bytes(B, I, J, ctypes.byref(need)))
        ws = torch.empty(max(need.value, 256), dtype=torch.uint8, device=X.device)
        out = torch.empty((2 * B, J), dtype=torch.float32, device=X.device)
        sz = torch.empty((B, I), dtype=torch.float32, device=X.device)
        perm = torch.empty((B, I), dtype=torch.int32, device=X.device)
        ck = torch.empty((B, J), dtype=torch.int32, device=X.device)
        _lib.check(lib.snntc_fc_forward_ex(_ptr(X), _ptr(W), pp, _ptr(out), _ptr(sz), _ptr(perm), _ptr(ck),
                                           B, I, J, w_rows, _ptr(ws), ws.numel(), _stream(X.device)))
    return out, sz, perm, ck


def init(device=None):
    """One-time set-up of a device (kernel attributes, the library's static scratch): call it before
    capturing library calls into a HIP graph.  device=None means the current device."""
    lib = _lib.load()
    if device is None:
        index = -1
    else:
        index = torch.device(device).index
        index = torch.cuda.current_device() if index is None else index
    _lib.check(lib.snntc_init(index))


def snnfc_static(X, W, Params, out=None):
    """snnfc through the entry point that allocates nothing: the scratch is a static device array
    inside the library (snntc_static_scratch_bytes()).  `out` may be a preallocated [2B,J] tensor.
    Calls on one GPU share that array: do not overlap them."""
    lib = _lib.load()
    X = _dev_f32(X, "X", 2)
    W = _dev_f32(W, "W", 2)
    p, pp = _params(Params, 6)
    B, I = X.shape
    w_rows, J = W.shape
    with torch.cuda.device(X.device):
        if out is None:
            out = torch.empty((2 * B, J), dtype=torch.float32, device=X.device)
        elif tuple(out.shape) != (2 * B, J) or out.dtype != torch.float32 or not out.is_contiguous():
            raise ValueError(f"out must be a contiguous float32 [{2 * B},{J}] tensor")
        _lib.check(lib.snntc_fc_forward_static(_ptr(X), _ptr(W), pp, _ptr(out), B, I, J, w_rows, _stream(X.device)))
    return out


def snnfc_grad(grad, X, W, Params, Y, want_dparams=True, want_dx=True, want_dw=True, first_half_grad=False):
    """Dense backward.  grad[2B,J], Y[2B,J] = forward output -> (dX[B,I], dW like W, dParams[6]).
    dParams is all zeros (Params is a constant).  A want_* flag set to False skips that gradient
    (None is returned in its place).  first_half_grad: grad may hold its first B rows only, which are
    the ones the op reads."""
    return _lib.native().fc_backward(grad, X, W, Params, Y, want_dx, want_dw, want_dparams, first_half_grad)


def snncv_output_dims(H, W, Params):
    lib = _lib.load()
    p, pp = _params(Params, 12)
    nh, nw = ctypes.c_int64(), ctypes.c_int64()
    _lib.check(lib.snntc_cv_output_dims(H, W, pp, ctypes.byref(nh), ctypes.byref(nw)))
    return nh.value, nw.value


def snncv(X, W, Params, return_aux=False, next_xpad=None, next_offset=(0, 0)):
    """Conv forward on the already padded / cropped NHWC input X[B,H,W,C]; W[Kh*Kw*C+bias,Kc]
    -> Y[2B,Nh,Nw,Kc].  With return_aux=True also returns per-patch (sorted_z, perm, causal_k).
    next_xpad[B,h,w,Kc], if given, also receives the spike times, output pixel (nh, nw) at its pixel
    (nh + next_offset[0], nw + next_offset[1]): the padded input of the conv layer that follows."""
    if not return_aux:
        return _lib.native().cv_forward(X, W, Params, next_xpad, next_offset[0], next_offset[1])
    lib = _lib.load()
    X = _dev_f32(X, "X", 4)
    W = _dev_f32(W, "W", 2)
    p, pp = _params(Params, 12)
    B, H, Wd, C = X.shape
    w_rows, Kc = W.shape
    Nh, Nw = snncv_output_dims(H, Wd, p)
    with torch.cuda.device(X.device):
        need = ctypes.c_size_t()
        _lib.check(lib.snntc_cv_forward_workspace_bytes(B, H, Wd, C, Kc, pp, ctypes.byref(need)))
        ws = torch.empty(max(need.value, 256), dtype=torch.uint8, device=X.device)
        out = torch.empty((2 * B, Nh, Nw, Kc), dtype=torch.float32, device=X.device)
        S, P = B * Nh * Nw, int(p[6]) * int(p[7]) * C
        sz = torch.empty((S, P), dtype=torch.float32, device=X.device)
        perm = torch.empty((S, P), dtype=torch.int32, device=X.device)
        ck = torch.empty((S, Kc), dtype=torch.int32, device=X.device)
        _lib.check(lib.snntc_cv_forward_ex(_ptr(X), _ptr(W), pp, _ptr(out), _ptr(sz), _ptr(perm), _ptr(ck),
                                           B, H, Wd, C, Kc, w_rows, _ptr(ws), ws.numel(), _stream(X.device)))
    return out, sz, perm, ck


def snncv_grad(grad, X, W, Params, Y, want_dparams=True, want_dx=True, want_dw=True, first_half_grad=False,
               crop=None):
    """Conv backward -> (dXpad like X, dW like W, dParams[12] of zeros, or None if not wanted).
    crop = (h, w, top, left): dX is only that window of the padded input's gradient, [B,h,w,C] (the
    gradient with respect to the image before its SAME padding)."""
    return _lib.native().cv_backward(grad, X, W, Params, Y, want_dx, want_dw, want_dparams, first_half_grad,
                                     None if crop is None else tuple(crop))


def _keep(ctx, X, W, Y, Params):
    ctx.save_for_backward(X, W, Y)
    ctx.params = np.array(Params, dtype=np.float32, copy=True)


def _layer_grads(op, ctx, grad, **how):
    X, W, Y = ctx.saved_tensors
    return op(grad, X, W, ctx.params, Y, want_dparams=False, want_dx=ctx.needs_input_grad[0],
              want_dw=ctx.needs_input_grad[1], **how)[:2]


class SnnFc(torch.autograd.Function):
    """Y = snnfc(X, W, Params) with the gradient the reference registers for "SnnFc"
    (SNN_TC_Modules.py:31-33): the backward op receives the full [2B,J] forward output."""

    @classmethod
    def apply(cls, X, W, Params):
        return _lib.native().fc_layer(X, W, Params, False)

    @staticmethod
    def forward(ctx, X, W, Params):
        Y = snnfc(X, W, Params)
        _keep(ctx, X, W, Y, Params)
        return Y

    @staticmethod
    def backward(ctx, grad):
        return *_layer_grads(snnfc_grad, ctx, grad), None


class SnnCv(torch.autograd.Function):
    """Y = snncv(Xpad, W, Params) with the gradient registered for "SnnCv" (SNN_TC_Modules.py:91-93)."""

    @classmethod
    def apply(cls, X, W, Params):
        return _lib.native().cv_layer(X, W, Params, False)

    @staticmethod
    def forward(ctx, X, W, Params):
        Y = snncv(X, W, Params)
        _keep(ctx, X, W, Y, Params)
        return Y

    @staticmethod
    def backward(ctx, grad):
        return *_layer_grads(snncv_grad, ctx, grad), None


class SnnFcTimes(torch.autograd.Function):
    """What SNN_dense.call returns (SNN_TC_Modules.py:73-75): the spike times Y[:B] of snnfc.  The full
    [2B,J] output is kept for the backward op, which then takes the [B,J] upstream gradient directly --
    slicing the output of SnnFc instead costs a zero fill and a copy of [2B,J] per backward pass."""

    @classmethod
    def apply(cls, X, W, Params):
        return _lib.native().fc_layer(X, W, Params, True)

    @staticmethod
    def forward(ctx, X, W, Params):
        Y = snnfc(X, W, Params)
        _keep(ctx, X, W, Y, Params)
        return Y[:X.shape[0]]

    @staticmethod
    def backward(ctx, grad):
        return *_layer_grads(snnfc_grad, ctx, grad, first_half_grad=True), None


class SnnCvTimes(torch.autograd.Function):
    """Spike times Y[:B] of snncv, as SNN_conv.call returns them (SNN_TC_Modules.py:168-170)."""

    @classmethod
    def apply(cls, X, W, Params):
        return _lib.native().cv_layer(X, W, Params, True)

    @staticmethod
    def forward(ctx, X, W, Params):
        Y = snncv(X, W, Params)
        _keep(ctx, X, W, Y, Params)
        return Y[:X.shape[0]]

    @staticmethod
    def backward(ctx, grad):
        return *_layer_grads(snncv_grad, ctx, grad, first_half_grad=True), None


class SnnCvSame(torch.autograd.Function):
    """SNN_conv with SAME padding as one differentiable step on the un-padded image x[B,H,W,C]: pad with
    MAX_SPIKE_TIME, snncv, and in the backward pass the gradient with respect to x itself (the op stores
    only that window of the padded gradient, so no separate crop runs).
      xpad      None: the padded tensor is made here (one pass).  Otherwise the layer's padded input
                buffer, already holding x in its interior (written there by the layer before, see
                next_xpad) and MAX_SPIKE_TIME on its border.
      next_xpad None, or the padded input buffer of the conv layer that follows: the spike times are
                written there as well, at pixel offset next_offset."""

    @classmethod
    def apply(cls, x, W, Params, pads, xpad, next_xpad, next_offset):
        return _lib.native().cv_same(x, W, Params, pads[0], pads[1], pads[2], pads[3], xpad, next_xpad, next_offset[0],
                                     next_offset[1])

    @staticmethod
    def forward(ctx, x, W, Params, pads, xpad, next_xpad, next_offset):
        top, bottom, left, right = pads
        B, H, Wd, C = x.shape
        if xpad is None:
            xpad = pad_time(x, top, bottom, left, right, float(Params[0])) if any(pads) else x
        elif tuple(xpad.shape) != (B, top + H + bottom, left + Wd + right, C):
            raise ValueError(f"padded buffer {tuple(xpad.shape)} does not match input {tuple(x.shape)} and pads {pads}")
        Y = snncv(xpad, W, Params, next_xpad=next_xpad, next_offset=next_offset)
        _keep(ctx, xpad, W, Y, Params)
        ctx.crop = (H, Wd, top, left)
        return Y[:B]

    @staticmethod
    def backward(ctx, grad):
        return *_layer_grads(snncv_grad, ctx, grad, first_half_grad=True, crop=ctx.crop), None, None, None, None, None


def softmax_time_loss(times, label, want_loss=True, want_grad=True):
    """Per-sample cross-entropy of label[B,J] against softmax(-times[B,J]) and the gradient of its batch
    mean with respect to times, in one kernel (loss_func, SNN_TC_Modules.py:286-288).
    Returns (sample_loss[B] or None, dtimes[B,J] or None)."""
    return _lib.native().time_loss(times, label, want_loss, want_grad)


def sgd_update(params, grads, lr):
    """In place ``w -= lr * dw`` for every (w, dw) pair, all tensors in one launch: the SGD update of
    a training step (the reference hands it to the framework's optimizer, snntc/snntc-mnist.py:70)."""
    params, grads = list(params), list(grads)
    if len(params) != len(grads):
        raise ValueError(f"sgd_update: {len(params)} weight tensors but {len(grads)} gradients")
    if params:
        _lib.native().sgd_update(params, grads, lr)


class SoftmaxTimeLoss(torch.autograd.Function):
    """mean_b CE(label_b, softmax(-times_b)); the gradient is produced by the forward kernel."""

    @classmethod
    def apply(cls, times, label):
        return _lib.native().loss_layer(times, label)

    @staticmethod
    def forward(ctx, times, label):
        loss, grad = softmax_time_loss(times, label, want_grad=times.requires_grad)
        ctx.save_for_backward(*[] if grad is None else [grad])
        return loss.mean()

    @staticmethod
    def backward(ctx, upstream):
        return (ctx.saved_tensors[0] * upstream if ctx.saved_tensors else None), None


def min_pool(x, kernel, stride, pad, out_hw, pad_value=1e5, want_arg=True, next_xpad=None, next_offset=(0, 0)):
    """Earliest-spike pooling of NHWC spike times x[B,H,W,C] -> (y[B,Nh,Nw,C], arg or None).
    kernel = (Kh, Kw), stride = (Sh, Sw), pad = (top, left), out_hw = (Nh, Nw); pixels outside the
    image count as pad_value.  arg records, per output, the window position that attained the minimum.
    next_xpad[B,h,w,C], if given, also receives y at pixel offset next_offset (the padded input of the
    conv layer that follows)."""
    return _lib.native().min_pool(x, kernel[0], kernel[1], stride[0], stride[1], pad[0], pad[1], out_hw[0], out_hw[1],
                                  pad_value, want_arg, next_xpad, next_offset[0], next_offset[1])


def min_pool_grad(grad_y, arg, in_shape, kernel, stride, pad):
    """Gradient of min_pool with respect to its input: every pixel adds the gradients of the windows
    that recorded it."""
    lib = _lib.load()
    grad_y = _dev_f32(grad_y, "grad_y", 4)
    B, H, W, C = in_shape
    Nh, Nw = grad_y.shape[1], grad_y.shape[2]
    if tuple(arg.shape) != tuple(grad_y.shape) or arg.dtype != torch.int32 or not arg.is_contiguous():
        raise ValueError("arg must be the contiguous int32 tensor min_pool returned")
    with torch.cuda.device(grad_y.device):
        dx = torch.empty((B, H, W, C), dtype=torch.float32, device=grad_y.device)
        _lib.check(lib.snntc_min_pool_backward(_ptr(grad_y), _ptr(arg), _ptr(dx), B, H, W, C, kernel[0], kernel[1],
                                               stride[0], stride[1], pad[0], pad[1], Nh, Nw, _stream(grad_y.device)))
    return dx


class SnnMinPool(torch.autograd.Function):
    """SNN_maxpool2d on device tensors: min over the (implicitly padded) window, gradient to the
    position that attained it."""

    @classmethod
    def apply(cls, x, kernel, stride, pad, out_hw, pad_value, next_xpad=None, next_offset=(0, 0)):
        return _lib.native().min_pool_layer(x, kernel[0], kernel[1], stride[0], stride[1], pad[0], pad[1], out_hw[0], out_hw[1],
                                            pad_value, next_xpad, next_offset[0], next_offset[1])

    @staticmethod
    def forward(ctx, x, kernel, stride, pad, out_hw, pad_value, next_xpad, next_offset):
        y, arg = min_pool(x, kernel, stride, pad, out_hw, pad_value, want_arg=x.requires_grad, next_xpad=next_xpad,
                          next_offset=next_offset)
        ctx.geom = (tuple(x.shape), kernel, stride, pad)
        ctx.save_for_backward(*[] if arg is None else [arg])
        return y

    @staticmethod
    def backward(ctx, grad_y):
        dx = min_pool_grad(grad_y, ctx.saved_tensors[0], *ctx.geom) if ctx.saved_tensors else None
        return dx, None, None, None, None, None, None, None


def pad_time(x, top, bottom, left, right, value):
    """x[B,H,W,C] -> [B, top+H+bottom, left+W+right, C], the border filled with `value` (one pass)."""
    lib = _lib.load()
    x = _dev_f32(x, "x", 4)
    B, H, W, C = x.shape
    Hp, Wp = top + H + bottom, left + W + right
    with torch.cuda.device(x.device):
        xpad = torch.empty((B, Hp, Wp, C), dtype=torch.float32, device=x.device)
        _lib.check(lib.snntc_pad_time_forward(_ptr(x), _ptr(xpad), B, H, W, C, top, left, Hp, Wp, float(value),
                                              _stream(x.device)))
    return xpad


def pad_time_grad(dxpad, in_shape, top, left):
    """The gradient of pad_time: the H x W interior of dxpad."""
    lib = _lib.load()
    dxpad = _dev_f32(dxpad, "dxpad", 4)
    B, H, W, C = in_shape
    with torch.cuda.device(dxpad.device):
        dx = torch.empty((B, H, W, C), dtype=torch.float32, device=dxpad.device)
        _lib.check(lib.snntc_pad_time_backward(_ptr(dxpad), _ptr(dx), B, H, W, C, top, left, dxpad.shape[1],
                                               dxpad.shape[2], _stream(dxpad.device)))
    return dx


class SnnPadTime(torch.autograd.Function):
    """SAME padding of a conv layer's input with MAX_SPIKE_TIME, one kernel each way."""

    @classmethod
    def apply(cls, x, top, bottom, left, right, value):
        return _lib.native().pad_layer(x, top, bottom, left, right, value)

    @staticmethod
    def forward(ctx, x, top, bottom, left, right, value):
        ctx.geom = (tuple(x.shape), top, left)
        return pad_time(x, top, bottom, left, right, value)

    @staticmethod
    def backward(ctx, dxpad):
        return pad_time_grad(dxpad, *ctx.geom), None, None, None, None, None


def _function(cls, *args):
    return super(cls, cls).apply(*args)                     # torch.autograd.Function's own


#: the differentiable ops with the arguments of their native entry points, as torch.autograd.Function runs them
GENERAL = {
    "fc_layer": lambda X, W, Params, times: _function(SnnFcTimes if times else SnnFc, X, W, Params),
    "cv_layer": lambda X, W, Params, times: _function(SnnCvTimes if times else SnnCv, X, W, Params),
    "cv_same": lambda x, W, Params, top, bottom, left, right, xpad, next_xpad, ntop, nleft: _function(
        SnnCvSame, x, W, Params, (top, bottom, left, right), xpad, next_xpad, (ntop, nleft)),
    "min_pool_layer": lambda x, kh, kw, sh, sw, top, left, nh, nw, value, next_xpad, ntop, nleft: _function(
        SnnMinPool, x, (kh, kw), (sh, sw), (top, left), (nh, nw), value, next_xpad, (ntop, nleft)),
    "pad_layer": lambda x, top, bottom, left, right, value: _function(SnnPadTime, x, top, bottom, left, right, value),
    "loss_layer": lambda times, label: _function(SoftmaxTimeLoss, times, label),
}
