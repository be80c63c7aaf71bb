// Host path of the Python package: argument checks, output and scratch allocation, the C ABI calls and
// the autograd nodes of the ops, in one native call per op.
//
// What bounds the small calls is the host: a dense forward at one sample is three launches of 5-12 us,
// and the same call made through ctypes and torch.autograd.Function spent 15-25 us of interpreter time
// per op and as much again per backward node (784-800-800-10 at B=256: 348 us per training step for
// 215 us of kernels).  Here an op costs its launches plus 3-4 us.
//
// The library is reached through function pointers looked up in the very file _lib.py has loaded.
// Scratch comes from PyTorch's caching allocator per call: it is stream-ordered, belongs to the graph's
// pool while a stream is captured, and is safe with several threads and streams without a pool of ours.
// The GIL is released while an op runs.
//
// The nodes below know reverse mode over ordinary tensors.  Everything else PyTorch can hand an op -- forward-mode
// tangents, functorch's wrappers, tensors of Python modes, a tracer that has to see the call -- goes to the
// torch.autograd.Function of the same op in ops.py, which refuses or records it as any such function does (`plain`).
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/autograd.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <array>
#include <optional>
#include <string>
#include <vector>

#include "../../include/snntc.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ---- the library ---------------------------------------------------------------------------------------------------

#define SNNTC_BOUND(F)                                                                                             \
    F(snntc_last_error) F(snntc_fc_forward) F(snntc_fc_forward_workspace_bytes) F(snntc_fc_backward)               \
    F(snntc_fc_backward_workspace_bytes) F(snntc_cv_output_dims) F(snntc_cv_forward)                               \
    F(snntc_cv_forward_chained) F(snntc_cv_forward_workspace_bytes) F(snntc_cv_backward_cropped)                   \
    F(snntc_cv_backward_workspace_bytes) F(snntc_softmax_time_loss) F(snntc_sgd_update)                            \
    F(snntc_min_pool_forward) F(snntc_min_pool_forward_chained) F(snntc_min_pool_backward)                         \
    F(snntc_pad_time_forward) F(snntc_pad_time_backward) F(snntc_encode_time) F(snntc_label_loss)                  \
    F(snntc_weight_cost_workspace_bytes) F(snntc_weight_cost_sums) F(snntc_weight_cost_grad) F(snntc_recipe_total)

struct Library {
#define SNNTC_FIELD(f) decltype(&::f) f = nullptr;
    SNNTC_BOUND(SNNTC_FIELD)
#undef SNNTC_FIELD
} lib;

PyObject* g_library_error = nullptr;   // snntc_amd._lib.SnntcLibraryError
PyObject* g_error = nullptr;           // snntc_amd._lib.SnntcError
PyObject* g_params = nullptr;          // snntc_amd._lib.params_array: any sequence -> contiguous float32 vector
PyObject* g_general = nullptr;         // snntc_amd.ops.GENERAL: name of a differentiable op -> its torch.autograd.Function

// Raises a Python exception of class `cls` from code that may run without the GIL (an autograd thread).
[[noreturn]] void raise_class(PyObject* cls, PyObject* (*args)(int, const std::string&), int status, const std::string& msg) {
    PyGILState_STATE gil = PyGILState_Ensure();
    PyObject* a = args(status, msg);
    if (a) PyErr_SetObject(cls, a);
    Py_XDECREF(a);
    python_error err;
    err.persist();
    PyGILState_Release(gil);
    throw std::move(err);
}

PyObject* message_args(int, const std::string& m) { return Py_BuildValue("(s)", m.c_str()); }
PyObject* status_args(int s, const std::string& m) { return Py_BuildValue("(is)", s, m.c_str()); }

// Maps a status code to the exception the reference's Python caller would see.
void check(int status) {
    if (status == SNNTC_OK) return;
    const std::string msg = lib.snntc_last_error();
    if (status == SNNTC_ERR_DIM_MISMATCH || status == SNNTC_ERR_TOO_LARGE || status == SNNTC_ERR_BAD_ARGUMENT)
        TORCH_CHECK_VALUE(false, msg);
    raise_class(g_error, status_args, status, msg);
}

// ---- tensors -------------------------------------------------------------------------------------------------------

std::string shape_text(const Tensor& t) {
    std::string s = "(";
    for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
    return s + (t.dim() == 1 ? ",)" : ")");
}

Tensor dev_f32(const Tensor& t, const char* name, int64_t ndim) {
    if (!t.is_cuda())
        raise_class(g_library_error, message_args, 0, std::string(name) + " lives on " + t.device().str() +
                    ": the SNN-TC ops run on a ROCm GPU only (no CPU fallback)");
    TORCH_CHECK_TYPE(t.scalar_type() == at::kFloat, name, " must be float32, got ", t.scalar_type());
    TORCH_CHECK_VALUE(t.dim() == ndim, name, " must have ", ndim, " dimensions, got shape ", shape_text(t));
    return t.contiguous();
}

float* f32(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor scratch(const Tensor& like, size_t bytes) {
    return at::empty({(int64_t)std::max<size_t>(bytes, 256)}, like.options().dtype(at::kByte));
}

Tensor empty(const Tensor& like, at::IntArrayRef sizes) { return at::empty(sizes, like.options()); }

// The first half of an op's [2B,...] output: the spike times.  It shares storage and version counter
// with the whole, so an in-place change of it is seen by the saved whole.
Tensor first_half(const Tensor& y, int64_t B) {
    at::AutoDispatchBelowADInplaceOrView guard;
    Tensor half = y.narrow(0, 0, B);
    torch::autograd::impl::set_version_counter(half, torch::autograd::impl::version_counter(y));
    return half;
}

bool wants_grad(const Tensor& a) { return at::GradMode::is_enabled() && a.requires_grad(); }
bool wants_grad(const Tensor& a, const Tensor& b) { return at::GradMode::is_enabled() && (a.requires_grad() || b.requires_grad()); }

// Whether the native nodes may stand for PyTorch's own machinery: no tangent to carry on, no wrapper without memory of
// its own, no mode, transform or tracer that has to see the operation.
bool plain(std::initializer_list<std::reference_wrapper<const Tensor>> tensors) {
    static const c10::DispatchKeySet special{
        c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
        c10::DispatchKey::ZeroTensor, c10::DispatchKey::Batched, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper};
    if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        return false;
    for (const Tensor& t : tensors)
        if (t.defined() && (t.key_set().has_any(special) || t._fw_grad(0).defined())) return false;
    return true;
}

// ---- the ops -------------------------------------------------------------------------------------------------------

using FcParams = std::array<float, 6>;
using CvParams = std::array<float, 12>;

Tensor fc_forward(const Tensor& x, const Tensor& w, const FcParams& p) {
    const int64_t B = x.size(0), I = x.size(1), rows = w.size(0), J = w.size(1);
    const c10::DeviceGuard guard(x.device());
    size_t need = 0;
    check(lib.snntc_fc_forward_workspace_bytes(B, I, J, &need));
    const Tensor ws = scratch(x, need), out = empty(x, {2 * B, J});
    check(lib.snntc_fc_forward(f32(x), f32(w), p.data(), f32(out), B, I, J, rows, ws.data_ptr(), ws.numel(), stream_of(x)));
    return out;
}

struct Grads { Tensor dx, dw, dp; };

Grads fc_backward(const Tensor& grad, const Tensor& x, const Tensor& w, const FcParams& p, const Tensor& y, bool want_dx,
                  bool want_dw, bool want_dp, bool first_half_grad) {
    const int64_t B = x.size(0), I = x.size(1), rows = w.size(0), J = w.size(1);
    TORCH_CHECK_VALUE(y.size(0) == 2 * B && y.size(1) == J && grad.size(1) == J, "Grad/Oldout batch should be 2 * batch: Y ",
                      shape_text(y), ", grad ", shape_text(grad), ", X ", shape_text(x), ", W ", shape_text(w));
    const c10::DeviceGuard guard(x.device());
    size_t need = 0;
    check(lib.snntc_fc_backward_workspace_bytes(B, I, J, &need));
    const Tensor ws = scratch(x, need);
    Grads g;
    if (want_dx) g.dx = empty(x, x.sizes());
    if (want_dw) g.dw = empty(w, w.sizes());
    if (want_dp) g.dp = empty(x, {6});
    // the op only ever reads rows [0,B) of grad, so a caller that holds just those rows passes them as is
    const int64_t grad_rows = first_half_grad && grad.size(0) == B ? 2 * B : grad.size(0);
    check(lib.snntc_fc_backward(f32(grad), f32(x), f32(w), p.data(), f32(y), f32(g.dx), f32(g.dw), f32(g.dp), B, I, J, rows,
                                grad_rows, ws.data_ptr(), ws.numel(), stream_of(x)));
    return g;
}

// Where an op also writes its spike times: pixel (nh + top, nw + left) of the next layer's padded input.
struct Feed { Tensor dst; int64_t top = 0, left = 0; };

Tensor feed_target(const Feed& feed, int64_t B, int64_t C, const char* what) {
    Tensor nx = dev_f32(feed.dst, "next_xpad", 4);
    TORCH_CHECK_VALUE(nx.size(0) == B && nx.size(3) == C, "next_xpad ", shape_text(nx), " does not match batch ", B, " / channels ", C);
    TORCH_CHECK_VALUE(nx.is_same(feed.dst), what, ": next_xpad must be contiguous");
    return nx;
}

// A kernel has written into `t` through its raw pointer: its version counter is advanced, so that autograd
// refuses a backward pass whose saved input has been overwritten by a later forward pass.
void written_behind_autograd(const Tensor& t) { t.unsafeGetTensorImpl()->bump_version(); }

Tensor cv_forward(const Tensor& x, const Tensor& w, const CvParams& p, const Feed& feed) {
    const int64_t B = x.size(0), H = x.size(1), W = x.size(2), C = x.size(3), rows = w.size(0), Kc = w.size(1);
    const c10::DeviceGuard guard(x.device());
    int64_t nh = 0, nw = 0;
    size_t need = 0;
    check(lib.snntc_cv_output_dims(H, W, p.data(), &nh, &nw));
    check(lib.snntc_cv_forward_workspace_bytes(B, H, W, C, Kc, p.data(), &need));
    const Tensor ws = scratch(x, need), out = empty(x, {2 * B, nh, nw, Kc});
    if (!feed.dst.defined()) {
        check(lib.snntc_cv_forward(f32(x), f32(w), p.data(), f32(out), B, H, W, C, Kc, rows, ws.data_ptr(), ws.numel(), stream_of(x)));
        return out;
    }
    const Tensor nx = feed_target(feed, B, Kc, "snncv");
    check(lib.snntc_cv_forward_chained(f32(x), f32(w), p.data(), f32(out), f32(nx), nx.size(1), nx.size(2), feed.top, feed.left,
                                       B, H, W, C, Kc, rows, ws.data_ptr(), ws.numel(), stream_of(x)));
    written_behind_autograd(nx);
    return out;
}

struct Window { int64_t h = 0, w = 0, top = 0, left = 0; };

Grads cv_backward(const Tensor& grad, const Tensor& x, const Tensor& w, const CvParams& p, const Tensor& y, bool want_dx,
                  bool want_dw, bool want_dp, bool first_half_grad, const Window* crop) {
    const int64_t B = x.size(0), H = x.size(1), W = x.size(2), C = x.size(3), rows = w.size(0), Kc = w.size(1);
    TORCH_CHECK_VALUE(y.size(0) == 2 * B && grad.sizes().slice(1) == y.sizes().slice(1) && y.size(3) == Kc,
                      "Grad/Oldout batch should be 2 * batch: Y ", shape_text(y), ", grad ", shape_text(grad), ", X ",
                      shape_text(x), ", W ", shape_text(w));
    const c10::DeviceGuard guard(x.device());
    size_t need = 0;
    check(lib.snntc_cv_backward_workspace_bytes(B, H, W, C, Kc, p.data(), &need));
    const Tensor ws = scratch(x, need);
    const Window win = crop ? *crop : Window{H, W, 0, 0};
    Grads g;
    if (want_dx) g.dx = empty(x, {B, win.h, win.w, C});
    if (want_dw) g.dw = empty(w, w.sizes());
    if (want_dp) g.dp = empty(x, {12});
    const int64_t grad_rows = first_half_grad && grad.size(0) == B ? 2 * B : grad.size(0);
    check(lib.snntc_cv_backward_cropped(f32(grad), f32(x), f32(w), p.data(), f32(y), f32(g.dx), win.h, win.w, win.top, win.left,
                                        f32(g.dw), f32(g.dp), B, H, W, C, Kc, rows, grad_rows, ws.data_ptr(), ws.numel(),
                                        stream_of(x)));
    return g;
}

struct Pads { int64_t top = 0, bottom = 0, left = 0, right = 0; };

Tensor pad_time(const Tensor& x, const Pads& pad, float value) {
    const int64_t B = x.size(0), H = x.size(1), W = x.size(2), C = x.size(3);
    const int64_t Hp = pad.top + H + pad.bottom, Wp = pad.left + W + pad.right;
    const c10::DeviceGuard guard(x.device());
    const Tensor out = empty(x, {B, Hp, Wp, C});
    check(lib.snntc_pad_time_forward(f32(x), f32(out), B, H, W, C, pad.top, pad.left, Hp, Wp, value, stream_of(x)));
    return out;
}

struct PoolShape { int64_t kh, kw, sh, sw, top, left, nh, nw; float pad_value; };

struct Pooled { Tensor y, arg; };

Pooled min_pool(const Tensor& x, const PoolShape& s, bool want_arg, const Feed& feed) {
    const int64_t B = x.size(0), H = x.size(1), W = x.size(2), C = x.size(3);
    const c10::DeviceGuard guard(x.device());
    Pooled r;
    r.y = empty(x, {B, s.nh, s.nw, C});
    if (want_arg) r.arg = at::empty({B, s.nh, s.nw, C}, x.options().dtype(at::kInt));
    int32_t* arg = want_arg ? static_cast<int32_t*>(r.arg.data_ptr()) : nullptr;
    if (!feed.dst.defined()) {
        check(lib.snntc_min_pool_forward(f32(x), f32(r.y), arg, B, H, W, C, s.kh, s.kw, s.sh, s.sw, s.top, s.left, s.nh, s.nw,
                                         s.pad_value, stream_of(x)));
        return r;
    }
    const Tensor nx = feed_target(feed, B, C, "min_pool");
    check(lib.snntc_min_pool_forward_chained(f32(x), f32(r.y), arg, f32(nx), nx.size(1), nx.size(2), feed.top, feed.left, B, H, W,
                                             C, s.kh, s.kw, s.sh, s.sw, s.top, s.left, s.nh, s.nw, s.pad_value, stream_of(x)));
    written_behind_autograd(nx);
    return r;
}

struct LossOut { Tensor loss, grad; };

LossOut time_loss(const Tensor& times, const Tensor& label, bool want_loss, bool want_grad) {
    TORCH_CHECK_VALUE(times.sizes() == label.sizes(), "loss: times ", shape_text(times), " and label ", shape_text(label),
                      " differ in shape");
    const c10::DeviceGuard guard(times.device());
    LossOut r;
    if (want_loss) r.loss = empty(times, {times.size(0)});
    if (want_grad) r.grad = empty(times, times.sizes());
    check(lib.snntc_softmax_time_loss(f32(times), f32(label), f32(r.loss), f32(r.grad), times.size(0), times.size(1),
                                      stream_of(times)));
    return r;
}

// ---- autograd nodes ------------------------------------------------------------------------------------------------

template <typename N>
Tensor with_history(Tensor out, const std::shared_ptr<N>& node) {
    torch::autograd::set_history(out, node);
    return out;
}

template <typename N>
std::shared_ptr<N> make_node(std::initializer_list<std::reference_wrapper<const Tensor>> inputs) {
    std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
    torch::autograd::edge_list edges;
    for (const Tensor& t : inputs) edges.push_back(torch::autograd::impl::gradient_edge(t));
    node->set_next_edges(std::move(edges));
    return node;
}

struct LayerNode : public Node {
    SavedVariable x, w, y;
    void save(const Tensor& x_, const Tensor& w_, const Tensor& y_) {
        x = SavedVariable(x_, false); w = SavedVariable(w_, false); y = SavedVariable(y_, false);
    }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        x.reset_data(); w.reset_data(); y.reset_data();
    }
};

struct FcNode : public LayerNode {
    FcParams params;
    bool first_half;                    // the upstream gradient has the rows of the spike times only
    std::string name() const override { return "SnnFcBackward"; }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(2);
        if (!grads[0].defined()) return out;
        const Tensor X = x.unpack(), Wt = w.unpack(), Y = y.unpack();
        at::AutoGradMode no_grad(false);
        Grads g = fc_backward(dev_f32(grads[0], "grad", 2), X, Wt, params, Y, task_should_compute_output(0),
                              task_should_compute_output(1), false, first_half);
        out[0] = g.dx; out[1] = g.dw;
        return out;
    }
};

struct CvNode : public LayerNode {
    CvParams params;
    bool first_half;
    std::optional<Window> crop;
    std::string name() const override { return "SnnCvBackward"; }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(2);
        if (!grads[0].defined()) return out;
        const Tensor X = x.unpack(), Wt = w.unpack(), Y = y.unpack();
        at::AutoGradMode no_grad(false);
        Grads g = cv_backward(dev_f32(grads[0], "grad", 4), X, Wt, params, Y, task_should_compute_output(0),
                              task_should_compute_output(1), false, first_half, crop ? &*crop : nullptr);
        out[0] = g.dx; out[1] = g.dw;
        return out;
    }
};

struct PoolNode : public Node {
    SavedVariable arg;
    PoolShape shape;
    std::array<int64_t, 4> in;
    std::string name() const override { return "SnnMinPoolBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        arg.reset_data();
    }
    variable_list apply(variable_list&& grads) override;
};

struct PadNode : public Node {
    std::array<int64_t, 4> in;
    int64_t top, left;
    std::string name() const override { return "SnnPadTimeBackward"; }
    variable_list apply(variable_list&& grads) override;
};

struct LossNode : public Node {
    SavedVariable grad;
    std::string name() const override { return "SoftmaxTimeLossBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        grad.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        if (!grads[0].defined()) return variable_list(1);
        return {grad.unpack() * grads[0]};                  // (differentiable in the upstream factor)
    }
};

Tensor min_pool_grad(const Tensor& gy, const Tensor& arg, const std::array<int64_t, 4>& in, const PoolShape& s) {
    TORCH_CHECK_VALUE(arg.sizes() == gy.sizes() && arg.scalar_type() == at::kInt && arg.is_contiguous(),
                      "arg must be the contiguous int32 tensor min_pool returned");
    const c10::DeviceGuard guard(gy.device());
    const Tensor dx = empty(gy, {in[0], in[1], in[2], in[3]});
    check(lib.snntc_min_pool_backward(f32(gy), static_cast<int32_t*>(arg.data_ptr()), f32(dx), in[0], in[1], in[2], in[3], s.kh, s.kw,
                                      s.sh, s.sw, s.top, s.left, gy.size(1), gy.size(2), stream_of(gy)));
    return dx;
}

Tensor pad_time_grad(const Tensor& dxpad, const std::array<int64_t, 4>& in, int64_t top, int64_t left) {
    const c10::DeviceGuard guard(dxpad.device());
    const Tensor dx = empty(dxpad, {in[0], in[1], in[2], in[3]});
    check(lib.snntc_pad_time_backward(f32(dxpad), f32(dx), in[0], in[1], in[2], in[3], top, left, dxpad.size(1), dxpad.size(2),
                                      stream_of(dxpad)));
    return dx;
}

variable_list PoolNode::apply(variable_list&& grads) {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!grads[0].defined() || !task_should_compute_output(0)) return variable_list(1);
    const Tensor a = arg.unpack();
    at::AutoGradMode no_grad(false);
    return {min_pool_grad(dev_f32(grads[0], "grad_y", 4), a, in, shape)};
}

variable_list PadNode::apply(variable_list&& grads) {
    if (!grads[0].defined() || !task_should_compute_output(0)) return variable_list(1);
    at::AutoGradMode no_grad(false);
    return {pad_time_grad(dev_f32(grads[0], "dxpad", 4), in, top, left)};
}

// `times`: hand out the spike times Y[:B] rather than the whole [2B,...] output.
Tensor fc_layer(const Tensor& x_in, const Tensor& w_in, const FcParams& p, bool times) {
    const Tensor x = dev_f32(x_in, "X", 2), w = dev_f32(w_in, "W", 2);
    Tensor y;
    {
        at::AutoGradMode no_grad(false);
        y = fc_forward(x, w, p);
    }
    Tensor out = times ? first_half(y, x.size(0)) : y;
    if (!wants_grad(x, w)) return out;
    auto node = make_node<FcNode>({x, w});
    node->params = p; node->first_half = times;
    // the whole output is handed out as it is: it is saved as a detached alias, or it would keep itself alive
    node->save(x, w, times ? y : y.detach());
    return with_history(out, node);
}

Tensor cv_layer(const Tensor& x_grad, const Tensor& x, const Tensor& w, const CvParams& p, bool times,
                const std::optional<Window>& crop, const Feed& feed) {
    Tensor y;
    {
        at::AutoGradMode no_grad(false);
        y = cv_forward(x, w, p, feed);
    }
    Tensor out = times ? first_half(y, x.size(0)) : y;
    if (!wants_grad(x_grad, w)) return out;
    auto node = make_node<CvNode>({x_grad, w});
    node->params = p; node->first_half = times; node->crop = crop;
    node->save(x, w, times ? y : y.detach());
    return with_history(out, node);
}

// SNN_conv with SAME padding on the un-padded image x: `xpad`, if given, is the layer's padded input buffer and
// already holds x.
Tensor cv_same(const Tensor& x_in, const Tensor& w_in, const CvParams& p, const Pads& pad, const Tensor& xpad_in, const Feed& feed) {
    const Tensor x = dev_f32(x_in, "X", 4), w = dev_f32(w_in, "W", 2);
    const int64_t B = x.size(0), H = x.size(1), W = x.size(2), C = x.size(3);
    Tensor xpad = xpad_in;
    if (!xpad.defined()) {
        at::AutoGradMode no_grad(false);
        xpad = pad.top || pad.bottom || pad.left || pad.right ? pad_time(x, pad, p[0]) : x;
    } else {
        TORCH_CHECK_VALUE((xpad.sizes() == at::IntArrayRef{B, pad.top + H + pad.bottom, pad.left + W + pad.right, C}),
                          "padded buffer ", shape_text(xpad), " does not match input ", shape_text(x), " and its pads");
        xpad = dev_f32(xpad, "X", 4);
    }
    return cv_layer(x, xpad, w, p, true, Window{H, W, pad.top, pad.left}, feed);
}

Tensor pool_layer(const Tensor& x_in, const PoolShape& s, const Feed& feed) {
    const Tensor x = dev_f32(x_in, "x", 4);
    const bool grad = wants_grad(x);
    Pooled r;
    {
        at::AutoGradMode no_grad(false);
        r = min_pool(x, s, grad, feed);
    }
    if (!grad) return r.y;
    auto node = make_node<PoolNode>({x});
    node->shape = s;
    node->in = {x.size(0), x.size(1), x.size(2), x.size(3)};
    node->arg = SavedVariable(r.arg, false);
    return with_history(r.y, node);
}

Tensor pad_layer(const Tensor& x_in, const Pads& pad, float value) {
    const Tensor x = dev_f32(x_in, "x", 4);
    Tensor out;
    {
        at::AutoGradMode no_grad(false);
        out = pad_time(x, pad, value);
    }
    if (!wants_grad(x)) return out;
    auto node = make_node<PadNode>({x});
    node->in = {x.size(0), x.size(1), x.size(2), x.size(3)};
    node->top = pad.top; node->left = pad.left;
    return with_history(out, node);
}

Tensor loss_layer(const Tensor& times_in, const Tensor& label_in) {
    const Tensor times = dev_f32(times_in, "times", 2), label = dev_f32(label_in, "label", 2);
    const bool grad = wants_grad(times);
    LossOut r;
    Tensor mean;
    {
        at::AutoGradMode no_grad(false);
        r = time_loss(times, label, true, grad);
        mean = r.loss.mean();
    }
    if (!grad) return mean;
    auto node = make_node<LossNode>({times});
    node->grad = SavedVariable(r.grad, false);
    return with_history(mean, node);
}

void sgd_update(const std::vector<Tensor>& ws, const std::vector<Tensor>& gs, float lr) {
    std::vector<float*> wp;
    std::vector<const float*> gp;
    std::vector<int64_t> n;
    std::vector<Tensor> keep;
    at::AutoGradMode no_grad(false);
    for (size_t i = 0; i < ws.size(); ++i) {
        const Tensor& w = ws[i];
        if (!(w.is_cuda() && w.scalar_type() == at::kFloat && w.is_contiguous()))
            raise_class(g_library_error, message_args, 0, "sgd_update: weight " + std::to_string(i) +
                        " must be a contiguous float32 tensor on a ROCm GPU");
        TORCH_CHECK_VALUE(gs[i].sizes() == w.sizes() && gs[i].scalar_type() == at::kFloat && gs[i].device() == w.device(),
                          "sgd_update: gradient ", i, " does not match its weight tensor");
        keep.push_back(gs[i].contiguous());
        wp.push_back(f32(w));
        gp.push_back(f32(keep.back()));
        n.push_back(w.numel());
    }
    const c10::DeviceGuard guard(ws[0].device());
    check(lib.snntc_sgd_update(wp.data(), gp.data(), n.data(), (int64_t)n.size(), lr, stream_of(ws[0])));
}

// ---- the example training recipe -------------------------------------------------------------------------------------

Tensor encode_time(const Tensor& image) {
    const Tensor x = image.contiguous();
    const c10::DeviceGuard guard(x.device());
    const Tensor z = empty(x, x.sizes());
    check(lib.snntc_encode_time(f32(x), f32(z), x.numel(), stream_of(x)));
    return z;
}

// Host arrays of the weight tensors the constraint cost runs over, and its device scratch.
struct CostArgs {
    std::vector<const float*> w;
    std::vector<int64_t> rows, cols;
    Tensor ws;
    explicit CostArgs(const std::vector<Tensor>& weights) {
        for (const Tensor& t : weights) {
            w.push_back(f32(t));
            rows.push_back(t.size(0));
            cols.push_back(t.size(1));
        }
    }
    int64_t count() const { return (int64_t)w.size(); }
    void sums(const Tensor& like, void* stream) {
        size_t need = 0;
        check(lib.snntc_weight_cost_workspace_bytes(rows.data(), cols.data(), count(), &need));
        ws = scratch(like, need);
        check(lib.snntc_weight_cost_sums(w.data(), rows.data(), cols.data(), count(), ws.data_ptr(), ws.numel(), stream));
    }
    void grad(float* const* g, float k, float k2, const float* upstream, bool accumulate, void* stream) {
        check(lib.snntc_weight_cost_grad(w.data(), g, rows.data(), cols.data(), count(), k, k2, upstream, accumulate, ws.data_ptr(),
                                         ws.numel(), stream));
    }
};

struct CostNode : public Node {
    std::vector<SavedVariable> weights;
    Tensor ws;
    float k, k2;
    std::string name() const override { return "ConstraintCostBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable& w : weights) w.reset_data();
        ws.reset();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(weights.size());
        if (!grads[0].defined()) return out;
        std::vector<Tensor> w;
        for (SavedVariable& s : weights) w.push_back(s.unpack());
        if (at::GradMode::is_enabled() || !plain({grads[0]})) {        // a graph of the gradient is wanted: differentiable ops
            for (size_t i = 0; i < w.size(); ++i) {
                if (!task_should_compute_output(i)) continue;
                const Tensor low = (1.0 - w[i].detach().sum(0)).ge(0).to(at::kFloat);
                out[i] = grads[0] * (low * (-k / (float)w[i].size(1)) + w[i] * (2.0f * k2 / (float)w[i].numel()));
            }
            return out;
        }
        const Tensor up = grads[0].contiguous();
        const c10::DeviceGuard guard(up.device());
        CostArgs args(w);
        args.ws = ws;
        std::vector<float*> g;
        for (size_t i = 0; i < w.size(); ++i) {
            if (task_should_compute_output(i)) out[i] = empty(w[i], w[i].sizes());
            g.push_back(f32(out[i]));
        }
        args.grad(g.data(), k, k2, f32(up), false, stream_of(up));
        return out;
    }
};

// The weight-constraint cost of contiguous float32 weight matrices on one device, differentiable.
Tensor constraint_cost(const std::vector<Tensor>& weights, float k, float k2) {
    const c10::DeviceGuard guard(weights[0].device());
    void* stream = stream_of(weights[0]);
    CostArgs args(weights);
    Tensor total;
    bool grad = false;
    {
        at::AutoGradMode no_grad(false);
        args.sums(weights[0], stream);
        total = empty(weights[0], {});
        check(lib.snntc_recipe_total(args.rows.data(), args.cols.data(), args.count(), k, k2, nullptr, nullptr, 0, f32(total), nullptr,
                                     args.ws.data_ptr(), args.ws.numel(), stream));
    }
    for (const Tensor& w : weights) grad = grad || wants_grad(w);
    if (!grad) return total;
    std::shared_ptr<CostNode> node(new CostNode(), torch::autograd::deleteNode);
    torch::autograd::edge_list edges;
    for (const Tensor& w : weights) {
        edges.push_back(torch::autograd::impl::gradient_edge(w));
        node->weights.emplace_back(w, false);
    }
    node->set_next_edges(std::move(edges));
    node->ws = args.ws; node->k = k; node->k2 = k2;
    return with_history(total, node);
}

// Loss, cost, count of correct samples and -- with `train` -- every gradient of one step: the data gradients
// through the engine from the loss kernel's dtimes, then the cost's added into each weight's .grad.
LossOut recipe_step(const Tensor& pred_in, const Tensor& labels_in, const std::vector<Tensor>& weights, float k, float k2, bool train) {
    const Tensor pred = dev_f32(pred_in, "predictions", 2);
    const int64_t B = pred.size(0), J = pred.size(1);
    const c10::DeviceGuard guard(pred.device());
    void* stream = stream_of(pred);
    Tensor sample_loss, dtimes, correct, total, n_correct;
    CostArgs args(weights);
    {
        at::AutoGradMode no_grad(false);
        const Tensor labels = labels_in.contiguous();
        sample_loss = empty(pred, {B});
        correct = at::empty({B}, pred.options().dtype(at::kInt));
        if (train) dtimes = empty(pred, pred.sizes());
        check(lib.snntc_label_loss(f32(pred), static_cast<int64_t*>(labels.data_ptr()), f32(sample_loss), f32(dtimes),
                                   static_cast<int32_t*>(correct.data_ptr()), B, J, stream));
    }
    if (train) torch::autograd::backward({pred}, {dtimes});
    at::AutoGradMode no_grad(false);
    args.sums(pred, stream);
    total = empty(pred, {});
    n_correct = at::empty({}, pred.options().dtype(at::kLong));
    check(lib.snntc_recipe_total(args.rows.data(), args.cols.data(), args.count(), k, k2, f32(sample_loss),
                                 static_cast<int32_t*>(correct.data_ptr()), B, f32(total), static_cast<int64_t*>(n_correct.data_ptr()),
                                 args.ws.data_ptr(), args.ws.numel(), stream));
    if (train) {
        std::vector<float*> g;
        std::vector<Tensor> keep;
        for (const Tensor& w : weights) {
            Tensor& wg = w.mutable_grad();
            if (!w.requires_grad()) { g.push_back(nullptr); continue; }
            if (!wg.defined()) {
                wg = at::zeros_like(w);
            } else if (!(wg.is_cuda() && wg.scalar_type() == at::kFloat && wg.is_contiguous() && wg.sizes() == w.sizes())) {
                wg = wg.to(w.options()).contiguous();
            }
            written_behind_autograd(wg);
            g.push_back(f32(wg));
        }
        args.grad(g.data(), k, k2, nullptr, true, stream);
    }
    return LossOut{total, n_correct};
}

// ---- Python arguments ----------------------------------------------------------------------------------------------

const Tensor& tensor_arg(PyObject* o, const char* name) {
    TORCH_CHECK_TYPE(THPVariable_Check(o), name, " must be a torch.Tensor");
    return THPVariable_Unpack(o);
}

Tensor optional_tensor(PyObject* o, const char* name) { return o == Py_None ? Tensor() : tensor_arg(o, name); }

int64_t int_arg(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}

float float_arg(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return (float)v;
}

bool bool_arg(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw python_error();
    return v != 0;
}

// A Params vector: read straight out of a float32 vector's buffer (what the layers keep), anything else is
// converted first.
template <size_t N>
std::array<float, N> params_arg(PyObject* o) {
    std::array<float, N> p;
    auto read = [&](PyObject* v) {
        Py_buffer b;
        if (PyObject_GetBuffer(v, &b, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) { PyErr_Clear(); return false; }
        const bool plain = b.format && b.format[0] == 'f' && b.format[1] == 0 && b.len == (Py_ssize_t)(N * sizeof(float));
        if (plain) memcpy(p.data(), b.buf, N * sizeof(float));
        PyBuffer_Release(&b);
        return plain;
    };
    if (read(o)) return p;
    PyObject* conv = PyObject_CallFunction(g_params, "On", o, (Py_ssize_t)N);     // raises ValueError on a wrong length
    if (!conv) throw python_error();
    const bool ok = read(conv);
    Py_DECREF(conv);
    TORCH_CHECK_VALUE(ok, "Params must hold ", N, " float32 values");
    return p;
}

struct NoGil {
    PyThreadState* state;
    NoGil() : state(PyEval_SaveThread()) {}
    ~NoGil() { PyEval_RestoreThread(state); }
};

void arity(Py_ssize_t got, Py_ssize_t want, const char* who) {
    TORCH_CHECK_TYPE(got == want, who, " takes ", want, " arguments, got ", got);
}

PyObject* wrap(const Tensor& t) {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}

PyObject* wrap3(const Tensor& a, const Tensor& b, const Tensor& c) {
    PyObject *pa = wrap(a), *pb = wrap(b), *pc = wrap(c);
    PyObject* t = pa && pb && pc ? PyTuple_Pack(3, pa, pb, pc) : nullptr;
    Py_XDECREF(pa); Py_XDECREF(pb); Py_XDECREF(pc);
    return t;
}

PyObject* wrap2(const Tensor& a, const Tensor& b) {
    PyObject *pa = wrap(a), *pb = wrap(b);
    PyObject* t = pa && pb ? PyTuple_Pack(2, pa, pb) : nullptr;
    Py_XDECREF(pa); Py_XDECREF(pb);
    return t;
}

Feed feed_arg(PyObject* dst, PyObject* top, PyObject* left) {
    return Feed{optional_tensor(dst, "next_xpad"), int_arg(top), int_arg(left)};
}

PyObject* general(const char* name, PyObject* const* a, Py_ssize_t n) {
    PyObject* f = PyDict_GetItemString(g_general, name);
    TORCH_CHECK(f, "no general path for ", name);
    return PyObject_Vectorcall(f, a, n, nullptr);
}

#define SNNTC_METHOD(name) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)

// fc_forward(X, W, params) -> Y[2B,J]
SNNTC_METHOD(py_fc_forward) {
    HANDLE_TH_ERRORS
    arity(n, 3, "fc_forward");
    const Tensor x = tensor_arg(a[0], "X"), w = tensor_arg(a[1], "W");
    const auto p = params_arg<6>(a[2]);
    Tensor out;
    {
        NoGil nogil;
        at::AutoGradMode no_grad(false);
        out = fc_forward(dev_f32(x, "X", 2), dev_f32(w, "W", 2), p);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// fc_layer(X, W, params, times) -> Y[:B] or Y, differentiable
SNNTC_METHOD(py_fc_layer) {
    HANDLE_TH_ERRORS
    arity(n, 4, "fc_layer");
    const Tensor x = tensor_arg(a[0], "X"), w = tensor_arg(a[1], "W");
    if (!plain({x, w})) return general("fc_layer", a, n);
    const auto p = params_arg<6>(a[2]);
    const bool times = bool_arg(a[3]);
    Tensor out;
    {
        NoGil nogil;
        out = fc_layer(x, w, p, times);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// fc_backward(grad, X, W, params, Y, want_dx, want_dw, want_dp, first_half_grad) -> (dX, dW, dP)
SNNTC_METHOD(py_fc_backward) {
    HANDLE_TH_ERRORS
    arity(n, 9, "fc_backward");
    const Tensor g = tensor_arg(a[0], "grad"), x = tensor_arg(a[1], "X"), w = tensor_arg(a[2], "W"), y = tensor_arg(a[4], "Y");
    const auto p = params_arg<6>(a[3]);
    const bool want_dx = bool_arg(a[5]), want_dw = bool_arg(a[6]), want_dp = bool_arg(a[7]), half = bool_arg(a[8]);
    Grads r;
    {
        NoGil nogil;
        at::AutoGradMode no_grad(false);
        r = fc_backward(dev_f32(g, "grad", 2), dev_f32(x, "X", 2), dev_f32(w, "W", 2), p, dev_f32(y, "Y", 2), want_dx, want_dw,
                        want_dp, half);
    }
    return wrap3(r.dx, r.dw, r.dp);
    END_HANDLE_TH_ERRORS
}

// cv_forward(X, W, params, next_xpad, top, left) -> Y[2B,Nh,Nw,Kc]
SNNTC_METHOD(py_cv_forward) {
    HANDLE_TH_ERRORS
    arity(n, 6, "cv_forward");
    const Tensor x = tensor_arg(a[0], "X"), w = tensor_arg(a[1], "W");
    const auto p = params_arg<12>(a[2]);
    const Feed feed = feed_arg(a[3], a[4], a[5]);
    Tensor out;
    {
        NoGil nogil;
        at::AutoGradMode no_grad(false);
        out = cv_forward(dev_f32(x, "X", 4), dev_f32(w, "W", 2), p, feed);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// cv_layer(X, W, params, times) -> Y[:B] or Y, differentiable
SNNTC_METHOD(py_cv_layer) {
    HANDLE_TH_ERRORS
    arity(n, 4, "cv_layer");
    const Tensor x = tensor_arg(a[0], "X"), w = tensor_arg(a[1], "W");
    if (!plain({x, w})) return general("cv_layer", a, n);
    const auto p = params_arg<12>(a[2]);
    const bool times = bool_arg(a[3]);
    Tensor out;
    {
        NoGil nogil;
        const Tensor xc = dev_f32(x, "X", 4);
        out = cv_layer(xc, xc, dev_f32(w, "W", 2), p, times, std::nullopt, Feed{});
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// cv_same(x, W, params, top, bottom, left, right, xpad, next_xpad, next_top, next_left) -> spike times, differentiable
SNNTC_METHOD(py_cv_same) {
    HANDLE_TH_ERRORS
    arity(n, 11, "cv_same");
    const Tensor x = tensor_arg(a[0], "X"), w = tensor_arg(a[1], "W");
    const auto p = params_arg<12>(a[2]);
    const Pads pad{int_arg(a[3]), int_arg(a[4]), int_arg(a[5]), int_arg(a[6])};
    const Tensor xpad = optional_tensor(a[7], "xpad");
    const Feed feed = feed_arg(a[8], a[9], a[10]);
    if (!plain({x, w, xpad, feed.dst})) return general("cv_same", a, n);
    Tensor out;
    {
        NoGil nogil;
        out = cv_same(x, w, p, pad, xpad, feed);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// cv_backward(grad, X, W, params, Y, want_dx, want_dw, want_dp, first_half_grad, crop) -> (dX, dW, dP)
SNNTC_METHOD(py_cv_backward) {
    HANDLE_TH_ERRORS
    arity(n, 10, "cv_backward");
    const Tensor g = tensor_arg(a[0], "grad"), x = tensor_arg(a[1], "X"), w = tensor_arg(a[2], "W"), y = tensor_arg(a[4], "Y");
    const auto p = params_arg<12>(a[3]);
    const bool want_dx = bool_arg(a[5]), want_dw = bool_arg(a[6]), want_dp = bool_arg(a[7]), half = bool_arg(a[8]);
    Window win;
    const bool cropped = a[9] != Py_None;
    if (cropped) {
        long long h, w2, t, l;
        if (!PyTuple_Check(a[9]) || !PyArg_ParseTuple(a[9], "LLLL", &h, &w2, &t, &l)) throw python_error();
        win = Window{h, w2, t, l};
    }
    Grads r;
    {
        NoGil nogil;
        at::AutoGradMode no_grad(false);
        r = cv_backward(dev_f32(g, "grad", 4), dev_f32(x, "X", 4), dev_f32(w, "W", 2), p, dev_f32(y, "Y", 4), want_dx, want_dw,
                        want_dp, half, cropped ? &win : nullptr);
    }
    return wrap3(r.dx, r.dw, r.dp);
    END_HANDLE_TH_ERRORS
}

PoolShape pool_arg(PyObject* const* a) {
    return PoolShape{int_arg(a[0]), int_arg(a[1]), int_arg(a[2]), int_arg(a[3]), int_arg(a[4]), int_arg(a[5]), int_arg(a[6]),
                     int_arg(a[7]), float_arg(a[8])};
}

// min_pool(x, kh, kw, sh, sw, top, left, nh, nw, pad_value, want_arg, next_xpad, next_top, next_left) -> (y, arg)
SNNTC_METHOD(py_min_pool) {
    HANDLE_TH_ERRORS
    arity(n, 14, "min_pool");
    const Tensor x = tensor_arg(a[0], "x");
    const PoolShape s = pool_arg(a + 1);
    const bool want_arg = bool_arg(a[10]);
    const Feed feed = feed_arg(a[11], a[12], a[13]);
    Pooled r;
    {
        NoGil nogil;
        at::AutoGradMode no_grad(false);
        r = min_pool(dev_f32(x, "x", 4), s, want_arg, feed);
    }
    return wrap2(r.y, r.arg);
    END_HANDLE_TH_ERRORS
}

// min_pool_layer(x, kh, kw, sh, sw, top, left, nh, nw, pad_value, next_xpad, next_top, next_left) -> y, differentiable
SNNTC_METHOD(py_min_pool_layer) {
    HANDLE_TH_ERRORS
    arity(n, 13, "min_pool_layer");
    const Tensor x = tensor_arg(a[0], "x");
    const PoolShape s = pool_arg(a + 1);
    const Feed feed = feed_arg(a[10], a[11], a[12]);
    if (!plain({x, feed.dst})) return general("min_pool_layer", a, n);
    Tensor out;
    {
        NoGil nogil;
        out = pool_layer(x, s, feed);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// pad_layer(x, top, bottom, left, right, value) -> padded, differentiable
SNNTC_METHOD(py_pad_layer) {
    HANDLE_TH_ERRORS
    arity(n, 6, "pad_layer");
    const Tensor x = tensor_arg(a[0], "x");
    if (!plain({x})) return general("pad_layer", a, n);
    const Pads pad{int_arg(a[1]), int_arg(a[2]), int_arg(a[3]), int_arg(a[4])};
    const float value = float_arg(a[5]);
    Tensor out;
    {
        NoGil nogil;
        out = pad_layer(x, pad, value);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// time_loss(times, label, want_loss, want_grad) -> (loss[B], dtimes)
SNNTC_METHOD(py_time_loss) {
    HANDLE_TH_ERRORS
    arity(n, 4, "time_loss");
    const Tensor t = tensor_arg(a[0], "times"), l = tensor_arg(a[1], "label");
    const bool want_loss = bool_arg(a[2]), want_grad = bool_arg(a[3]);
    LossOut r;
    {
        NoGil nogil;
        at::AutoGradMode no_grad(false);
        r = time_loss(dev_f32(t, "times", 2), dev_f32(l, "label", 2), want_loss, want_grad);
    }
    return wrap2(r.loss, r.grad);
    END_HANDLE_TH_ERRORS
}

// loss_layer(times, label) -> mean loss, differentiable in times
SNNTC_METHOD(py_loss_layer) {
    HANDLE_TH_ERRORS
    arity(n, 2, "loss_layer");
    const Tensor t = tensor_arg(a[0], "times"), l = tensor_arg(a[1], "label");
    if (!plain({t, l})) return general("loss_layer", a, n);
    Tensor out;
    {
        NoGil nogil;
        out = loss_layer(t, l);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// sgd_update(list of weights, list of gradients, lr)
SNNTC_METHOD(py_sgd_update) {
    HANDLE_TH_ERRORS
    arity(n, 3, "sgd_update");
    TORCH_CHECK_TYPE(PyList_Check(a[0]) && PyList_Check(a[1]), "sgd_update takes lists");
    std::vector<Tensor> ws, gs;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[0]); ++i) {
        PyObject* w = PyList_GET_ITEM(a[0], i);
        if (!THPVariable_Check(w))
            raise_class(g_library_error, message_args, 0, "sgd_update: weight " + std::to_string(i) +
                        " must be a contiguous float32 tensor on a ROCm GPU");
        ws.push_back(THPVariable_Unpack(w));
        gs.push_back(tensor_arg(PyList_GET_ITEM(a[1], i), "gradient"));
    }
    const float lr = float_arg(a[2]);
    {
        NoGil nogil;
        sgd_update(ws, gs, lr);
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

std::vector<Tensor> tensor_list(PyObject* o, const char* name) {
    TORCH_CHECK_TYPE(PyList_Check(o), name, " must be a list");
    std::vector<Tensor> v;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(o); ++i) v.push_back(tensor_arg(PyList_GET_ITEM(o, i), name));
    return v;
}

// plain(tensors...): whether the native entry points that have no general path may take them
SNNTC_METHOD(py_plain) {
    HANDLE_TH_ERRORS
    bool ok = plain({});
    for (Py_ssize_t i = 0; ok && i < n; ++i) ok = plain({tensor_arg(a[i], "argument")});
    return PyBool_FromLong(ok);
    END_HANDLE_TH_ERRORS
}

// encode_time(image) -> exp(1 - image) for a float32 device tensor
SNNTC_METHOD(py_encode_time) {
    HANDLE_TH_ERRORS
    arity(n, 1, "encode_time");
    const Tensor x = tensor_arg(a[0], "image");
    Tensor z;
    {
        NoGil nogil;
        at::AutoGradMode no_grad(false);
        z = encode_time(x);
    }
    return wrap(z);
    END_HANDLE_TH_ERRORS
}

// constraint_cost(weights, k, k2) -> scalar, differentiable
SNNTC_METHOD(py_constraint_cost) {
    HANDLE_TH_ERRORS
    arity(n, 3, "constraint_cost");
    const std::vector<Tensor> w = tensor_list(a[0], "weights");
    const float k = float_arg(a[1]), k2 = float_arg(a[2]);
    Tensor out;
    {
        NoGil nogil;
        out = constraint_cost(w, k, k2);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// recipe_step(predictions, labels, weights, k, k2, train) -> (loss, number of correct samples)
SNNTC_METHOD(py_recipe_step) {
    HANDLE_TH_ERRORS
    arity(n, 6, "recipe_step");
    const Tensor p = tensor_arg(a[0], "predictions"), l = tensor_arg(a[1], "labels");
    const std::vector<Tensor> w = tensor_list(a[2], "weights");
    const float k = float_arg(a[3]), k2 = float_arg(a[4]);
    const bool train = bool_arg(a[5]);
    LossOut r;
    {
        NoGil nogil;
        r = recipe_step(p, l, w, k, k2, train);
    }
    return wrap2(r.loss, r.grad);
    END_HANDLE_TH_ERRORS
}

// bind(path, SnntcLibraryError, SnntcError, params_array, general paths): looks the C ABI up in the library loaded from `path`
SNNTC_METHOD(py_bind) {
    HANDLE_TH_ERRORS
    arity(n, 5, "bind");
    const char* path = PyUnicode_AsUTF8(a[0]);
    if (!path) throw python_error();
    TORCH_CHECK_TYPE(PyDict_Check(a[4]), "bind takes a dict of general paths");
    for (int i = 1; i < 5; ++i) Py_INCREF(a[i]);
    Py_XDECREF(g_library_error); Py_XDECREF(g_error); Py_XDECREF(g_params); Py_XDECREF(g_general);
    g_library_error = a[1]; g_error = a[2]; g_params = a[3]; g_general = a[4];
    void* handle = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!handle) raise_class(g_library_error, message_args, 0, std::string("cannot load ") + path + ": " + dlerror());
    Library l;
#define SNNTC_LOOKUP(f)                                                                                            \
    l.f = reinterpret_cast<decltype(l.f)>(dlsym(handle, #f));                                                      \
    if (!l.f) raise_class(g_library_error, message_args, 0, std::string(path) + " lacks symbol " #f);
    SNNTC_BOUND(SNNTC_LOOKUP)
#undef SNNTC_LOOKUP
    lib = l;
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define SNNTC_ENTRY(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {SNNTC_ENTRY(bind), SNNTC_ENTRY(fc_forward), SNNTC_ENTRY(fc_layer), SNNTC_ENTRY(fc_backward),
                           SNNTC_ENTRY(cv_forward), SNNTC_ENTRY(cv_layer), SNNTC_ENTRY(cv_same), SNNTC_ENTRY(cv_backward),
                           SNNTC_ENTRY(min_pool), SNNTC_ENTRY(min_pool_layer), SNNTC_ENTRY(pad_layer), SNNTC_ENTRY(time_loss),
                           SNNTC_ENTRY(loss_layer), SNNTC_ENTRY(sgd_update), SNNTC_ENTRY(plain), SNNTC_ENTRY(encode_time),
                           SNNTC_ENTRY(constraint_cost), SNNTC_ENTRY(recipe_step), {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_binding", "Native host path of the SNN-TC ops.", -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) { return PyModule_Create(&g_module); }
