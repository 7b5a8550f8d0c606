// The host path from a torch tensor to a launch: allocation of the result and of the workspace, the current stream
// and the call of the C ABI, in one native call per layer.
//
// What bounds a decode-sized call is the host: a [4096 x 4096] product at one row is 3.8 us of GPU time, and the same
// steps taken in Python (module attributes, torch.empty, torch.cuda.device, current_stream, five ctypes calls) were
// 17 us of the 21 us a LowBitLinear call took.  The module is plain CPython (METH_FASTCALL, no argument parsing by
// keyword).  It holds no state but the addresses of the C ABI functions, which the ctypes binding hands over
// (`bind`), so that both always run the same library.
//
// Functions whose name says "or None" answer None for anything but the plain case (a tensor on another device, a
// dtype they do not know, a weight of another size): the Python code behind them then takes its own way and words
// the error.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>

#include "../../include/lowbit_abi.h"

namespace {

using at::Tensor;

struct Api {
    decltype(&lowbit_last_error) last_error = nullptr;
    decltype(&lowbit_blob_bytes) blob_bytes = nullptr;
    decltype(&lowbit_tileable) tileable = nullptr;
    decltype(&lowbit_linear_scratch_bytes) linear_scratch_bytes = nullptr;
    decltype(&lowbit_linear) linear = nullptr;
    decltype(&lowbit_gated_mlp) gated_mlp = nullptr;
    decltype(&lowbit_dequantize_rows) dequantize_rows = nullptr;
    decltype(&lowbit_dequantize) dequantize = nullptr;
    decltype(&lowbit_backward_ws) backward_ws = nullptr;
    decltype(&lowbit_backward_workspace_bytes) backward_workspace_bytes = nullptr;
    decltype(&lowbit_backward_ws_applies) backward_ws_applies = nullptr;
    decltype(&lowbit_experts_workspace_bytes) experts_workspace_bytes = nullptr;
    decltype(&lowbit_experts_forward) experts_forward = nullptr;
} api;

constexpr size_t WORKSPACE_CAP = (size_t)256 << 20;      // most that a product borrows for split-K partial sums

struct Failed : std::runtime_error {
    using std::runtime_error::runtime_error;
};

void check(int rc, const char *what) {
    if (rc != 0) throw Failed(std::string(what) + " failed (" + std::to_string(rc) + "): " + api.last_error());
}

int dtype_code(at::ScalarType t) {
    switch (t) {
    case at::kHalf: return LOWBIT_DT_F16;
    case at::kBFloat16: return LOWBIT_DT_BF16;
    case at::kFloat: return LOWBIT_DT_F32;
    default: return -1;
    }
}

void *current_stream(const Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// a tensor of this module's calls: strided, on the GPU
bool on_gpu(const Tensor &t) { return t.device().is_cuda() && t.layout() == at::kStrided; }

// whether the result has to carry a derivative with respect to t, which no call of this module gives it
bool differentiable(const Tensor &t) {
    return (t.requires_grad() && c10::GradMode::is_enabled()) || t._fw_grad(/*level=*/0).defined();
}

// w holds the packed [N, K] weight of this format on x's device
bool is_blob(const Tensor &w, const Tensor &x, int qtype, int64_t N, int64_t K) {
    if (w.device() != x.device() || w.layout() != at::kStrided || !w.is_contiguous()) return false;
    const at::ScalarType st = w.scalar_type();
    if (st != at::kByte && !(st == at::kBFloat16 && qtype == LOWBIT_QT_NF4)) return false;
    return (size_t)w.nbytes() == api.blob_bytes(qtype, N * K) && w.nbytes() > 0;
}

// y = x * dequant(w)^T (+ bias), in x's dtype; x contiguous [.., K] with M rows, not empty
Tensor product(const Tensor &x, const Tensor &w, const Tensor &bias, int qtype, int layout, int64_t M, int64_t N, int64_t K,
               at::IntArrayRef shape) {
    c10::DeviceGuard guard(x.device());
    Tensor y = at::empty(shape, x.options());
    const int dt = dtype_code(x.scalar_type());
    // the workspace comes from torch's caching allocator: ordered with the stream, no allocation in the steady state
    const size_t bytes = M <= 16 ? 0 : api.linear_scratch_bytes(qtype, layout, dt, M, N, K, WORKSPACE_CAP);
    const Tensor ws = bytes ? at::empty({(int64_t)bytes}, x.options().dtype(at::kByte)) : Tensor();
    check(api.linear(x.const_data_ptr(), w.const_data_ptr(), bias.defined() ? bias.const_data_ptr() : nullptr, y.data_ptr(), qtype,
                     layout, dt, M, N, K, bytes ? ws.data_ptr() : nullptr, bytes, current_stream(x)), "lowbit_linear");
    return y;
}

// Whether a small batch of float32 rows stays float32 (use_batch_forward of low_bit_linear.py)
bool batch_stays_f32(int qtype, int64_t M, int64_t N, int64_t K) {
    if (M <= 1 || K % 128) return false;
    if (qtype != LOWBIT_QT_SYM_INT4 && qtype != LOWBIT_QT_ASYM_INT4 && qtype != LOWBIT_QT_FP8_E4M3) return false;
    return M <= 48 || (M <= 64 && K % 256 == 0 && N % 64 == 0);
}

int device_layout(int qtype, int64_t N, int64_t K) {
    return api.tileable(qtype, N, K) ? LOWBIT_LAYOUT_TILED : LOWBIT_LAYOUT_GGML;
}

at::DimVector with_last(const Tensor &x, int64_t last) {
    at::DimVector shape(x.sizes().begin(), x.sizes().end());
    shape.back() = last;
    return shape;
}

// LowBitLinear at inference on a GPU-resident weight; an undefined tensor when this is not the plain case
Tensor linear(const Tensor &x_in, const Tensor &w, const Tensor &bias, int qtype, int64_t N, bool conver_to_half) {
    if (!on_gpu(x_in) || x_in.dim() < 1 || x_in.numel() == 0 || dtype_code(x_in.scalar_type()) < 0) return {};
    const int64_t K = x_in.size(-1), M = x_in.numel() / K;
    if (!is_blob(w, x_in, qtype, N, K)) return {};
    if (bias.defined() && (bias.scalar_type() != x_in.scalar_type() || bias.device() != x_in.device() || bias.numel() != N || !bias.is_contiguous() ||
                           differentiable(bias))) return {};
    const Tensor x = x_in.is_contiguous() ? x_in : x_in.contiguous();
    const int layout = device_layout(qtype, N, K);
    const auto shape = with_last(x, N);
    if (x.scalar_type() == at::kFloat && conver_to_half && M > 1 && !batch_stays_f32(qtype, M, N, K)) {
        Tensor y = product(x.to(at::kHalf), w, Tensor(), qtype, layout, M, N, K, shape).to(at::kFloat);
        if (bias.defined()) y.add_(bias);
        return y;
    }
    return product(x, w, bias, qtype, layout, M, N, K, shape);
}

// ---- training: the same product below trained parameters
//
// What bounded a small step was the host: a layer's forward and backward took some 110 us of Python, ctypes and the
// interpreter lock taken in autograd's thread, around 20 us of GPU time (77 rows on [1200 x 1024]).

// no transform (vmap, grad), trace or dispatch mode that wants to see the operators
bool nothing_watches(const Tensor &t) {
    using c10::DispatchKey;
    const c10::DispatchKeySet on = c10::impl::tls_local_dispatch_key_set().included_;
    if (on.has(DispatchKey::FuncTorchDynamicLayerFrontMode) || on.has(DispatchKey::Tracer) || on.has(DispatchKey::Functionalize) ||
        c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
    return !t.key_set().has_any(c10::DispatchKeySet({DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                                     DispatchKey::Batched, DispatchKey::Functionalize}));
}

// The gradient that flows on to x.  A node and not a torch::autograd::Function: it holds the weight as MatMulLowBit's context
// does, as it is when the backward runs, past saved-tensor hooks and through repeated backwards.
struct ProductBackward : public torch::autograd::Node {
    Tensor w;
    int qtype = 0, layout = 0;
    int64_t N = 0, K = 0;
    at::ScalarType dtype = at::kHalf;
    at::DimVector x_shape;

    std::string name() const override { return "MatMulLowBitBackward"; }

    torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
        if (!task_should_compute_output(0)) return {Tensor()};
        // (a gradient that a function above left out counts as zeros, as autograd functions in Python are given it)
        const Tensor grad = grads[0].defined() ? grads[0].to(dtype).reshape({-1, N})
                                               : at::zeros({c10::multiply_integers(x_shape) / K, N}, w.options().dtype(dtype));
        const int64_t M = grad.size(0);
        c10::DeviceGuard guard(grad.device());
        if (!is_blob(w, grad, qtype, N, K)) throw Failed("the low-bit weight is not where the forward found it");
        const int dt = dtype_code(dtype);
        void *const stream = current_stream(grad);
        const bool tracked = differentiable(grad) || !nothing_watches(grad);
        const size_t bytes = tracked ? 0 : api.backward_workspace_bytes(qtype, M, N, K);
        if (!tracked && api.backward_ws_applies(qtype, layout, dt, M, N, K, bytes)) {
            const Tensor g = grad.contiguous();
            if ((((uintptr_t)g.const_data_ptr() | (uintptr_t)w.const_data_ptr()) & 15) == 0) {
                Tensor gx = at::empty(x_shape, g.options());
                const Tensor ws = bytes ? at::empty({(int64_t)bytes}, g.options().dtype(at::kByte)) : Tensor();
                check(api.backward_ws(g.const_data_ptr(), w.const_data_ptr(), gx.data_ptr(), qtype, dt, M, N, K,
                                      bytes ? ws.data_ptr() : nullptr, bytes, stream), "lowbit_backward");
                return {gx};
            }
        }
        // (tracked: a second derivative, a tangent or a transform over the backward goes through the dense product)
        const Tensor dense = at::empty({N, K}, w.options().dtype(dtype));
        check(api.dequantize(w.const_data_ptr(), dense.data_ptr(), qtype, N, K, layout, dt, stream), "lowbit_dequantize");
        return {at::matmul(grad, dense).view(x_shape)};
    }
};

// LowBitLinear in training on a 16-bit x that wants a gradient, where the weight and bias want none; an undefined tensor when
// this is not the plain case
Tensor linear_train(const Tensor &x_in, const Tensor &w, const Tensor &bias, int qtype, int64_t N) {
    if (!on_gpu(x_in) || x_in.dim() < 1 || x_in.numel() == 0 || !x_in.requires_grad() || !c10::GradMode::is_enabled()) return {};
    const int dt = dtype_code(x_in.scalar_type());
    const int64_t K = x_in.size(-1), M = x_in.numel() / K;
    if ((dt != LOWBIT_DT_F16 && dt != LOWBIT_DT_BF16) || !nothing_watches(x_in) || x_in._fw_grad(/*level=*/0).defined() ||
        !is_blob(w, x_in, qtype, N, K) || w.requires_grad()) return {};
    if (bias.defined() && (bias.scalar_type() != x_in.scalar_type() || bias.device() != x_in.device() || bias.numel() != N || !bias.is_contiguous() ||
                           bias.requires_grad() || differentiable(bias))) return {};
    Tensor y;
    auto node = std::shared_ptr<ProductBackward>(new ProductBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(x_in));
    node->w = w;
    node->qtype = qtype;
    node->layout = device_layout(qtype, N, K);
    node->N = N;
    node->K = K;
    node->dtype = x_in.scalar_type();
    node->x_shape.assign(x_in.sizes().begin(), x_in.sizes().end());
    {
        c10::AutoGradMode no_grad(false);
        const Tensor x = x_in.detach().contiguous();
        y = product(x, w, bias, qtype, node->layout, M, N, K, with_last(x, N));
    }
    torch::autograd::set_history(y, node);
    return y;
}

// act(x Wg^T) * (x Wu^T) for 16-bit x and tiled weights; an undefined tensor when this is not the plain case
Tensor gated(const Tensor &x_in, const Tensor &wg, const Tensor &wu, int qtype, int64_t N, int act) {
    if (!on_gpu(x_in) || x_in.dim() < 1 || x_in.numel() == 0) return {};
    const int dt = dtype_code(x_in.scalar_type());
    if (dt != LOWBIT_DT_F16 && dt != LOWBIT_DT_BF16) return {};
    const int64_t K = x_in.size(-1), M = x_in.numel() / K;
    if (!is_blob(wg, x_in, qtype, N, K) || !is_blob(wu, x_in, qtype, N, K) || !api.tileable(qtype, N, K)) return {};
    const Tensor x = x_in.is_contiguous() ? x_in : x_in.contiguous();
    c10::DeviceGuard guard(x.device());
    Tensor y = at::empty(with_last(x, N), x.options());
    check(api.gated_mlp(x.const_data_ptr(), wg.const_data_ptr(), wu.const_data_ptr(), y.data_ptr(), qtype, dt, M, N, K, act,
                          current_stream(x)), "lowbit_gated_mlp");
    return y;
}

// rows ids[i] of the dequantized [N, K] table, in `dtype`; an undefined tensor when this is not the plain case
Tensor embedding(const Tensor &ids_in, const Tensor &w, int qtype, int64_t N, int64_t K, at::ScalarType dtype) {
    if (!on_gpu(ids_in) || ids_in.numel() == 0 || ids_in.scalar_type() != at::kLong || !is_blob(w, ids_in, qtype, N, K)) return {};
    const int dt = dtype_code(dtype);
    if (dt < 0) return {};
    const Tensor ids = ids_in.contiguous();
    c10::DeviceGuard guard(ids.device());
    at::DimVector shape(ids.sizes().begin(), ids.sizes().end());
    shape.push_back(K);
    Tensor y = at::empty(shape, ids.options().dtype(dtype));
    check(api.dequantize_rows(w.const_data_ptr(), ids.const_data_ptr<int64_t>(), ids.numel(), y.data_ptr(), qtype, N, K,
                              device_layout(qtype, N, K), dt, current_stream(ids)), "lowbit_dequantize_rows");
    return y;
}

// a table of n weight pointers in x's device memory
bool is_table(const Tensor &t, const Tensor &x, int64_t n) {
    return t.device() == x.device() && t.layout() == at::kStrided && t.scalar_type() == at::kLong && t.numel() == n && t.is_contiguous();
}

// the experts of a mixture-of-experts block on x [tokens, hidden]; tables: one weight pointer per expert, on x's device.
// The caller has checked what the pointers lead to: gate, up [inter, hidden] and down [hidden, inter] weights of one qtype.
Tensor experts(const Tensor &x_in, const Tensor &ids_in, const Tensor &weight_in, const Tensor &gates, const Tensor &ups,
               const Tensor &downs, int qtype, int64_t hidden, int64_t inter, int act) {
    if (!on_gpu(x_in) || x_in.dim() != 2 || x_in.size(1) != hidden || ids_in.dim() != 2 || ids_in.size(0) != x_in.size(0) ||
        ids_in.numel() == 0 || !at::isIntegralType(ids_in.scalar_type(), /*includeBool=*/false) || weight_in.sizes() != ids_in.sizes() ||
        ids_in.device() != x_in.device() || weight_in.device() != x_in.device() || !is_table(gates, x_in, gates.numel()) ||
        !is_table(ups, x_in, gates.numel()) || !is_table(downs, x_in, gates.numel()) || differentiable(weight_in)) return {};
    const int dt = dtype_code(x_in.scalar_type()), wdt = dtype_code(weight_in.scalar_type());
    if ((dt != LOWBIT_DT_F16 && dt != LOWBIT_DT_BF16) || wdt < 0) return {};
    const int64_t tokens = ids_in.size(0), top_k = ids_in.size(1), n_exp = gates.numel();
    const size_t bytes = top_k > 64 || n_exp > 4096 ? 0 : api.experts_workspace_bytes(tokens, (int)top_k, (int)n_exp, hidden, inter);
    if (!bytes) return {};                               // more than the library takes
    const Tensor x = x_in.contiguous(), ids = ids_in.to(at::kLong).contiguous(), weight = weight_in.contiguous();
    c10::DeviceGuard guard(x.device());
    const Tensor ws = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
    Tensor y = at::empty({tokens, hidden}, x.options());
    check(api.experts_forward(x.const_data_ptr(), ids.const_data_ptr<int64_t>(), weight.const_data_ptr(), wdt, tokens, (int)top_k,
                              (int)n_exp, (const void *const *)gates.const_data_ptr(), (const void *const *)ups.const_data_ptr(),
                              (const void *const *)downs.const_data_ptr(), ws.data_ptr(), bytes, y.data_ptr(), qtype, dt, hidden, inter,
                              act, current_stream(x)), "lowbit_experts_forward");
    return y;
}

// ---- large copies between pageable host memory and the GPU, through two pinned buffers
//
// A pageable copy by the runtime ran at 29 GB/s up and, into memory the process has not touched yet, 7.5 GB/s down
// (the bus: 57).  Here a chunk crosses the bus while all cores copy the one before or after it between pageable and
// pinned memory: [11008 x 4096] float16 up 3.2 -> 2.0 ms, its sym_int4 blob down 1.5 (fresh memory: 3.4) -> 0.6 ms.  The buffers are torch's
// (its caching allocator for pinned memory: kept between calls, at most two chunks per call in flight, safe with
// several threads and streams).  Smaller tensors are left to Tensor.to.
constexpr int64_t COPY_CHUNK = (int64_t)4 << 20;

struct Staging {
    c10::Stream stream;
    Tensor buffer[2];
    c10::Event done[2] = {c10::Event(c10::DeviceType::CUDA), c10::Event(c10::DeviceType::CUDA)};
    explicit Staging(c10::Device device) : stream(c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getStream(device)) {
        for (Tensor &b : buffer) b = at::empty({COPY_CHUNK}, at::TensorOptions().dtype(at::kByte).pinned_memory(true));
    }
};

Tensor as_bytes(const Tensor &t) {                       // the storage of a contiguous tensor as uint8 [nbytes]
    return at::empty({0}, t.options().dtype(at::kByte)).set_(t.storage(), t.storage_offset() * (int64_t)t.itemsize(), {(int64_t)t.nbytes()}, {1});
}

bool copies_in_chunks(const Tensor &t, bool gpu) {
    return t.layout() == at::kStrided && (gpu ? t.device().is_cuda() : t.device().is_cpu() && !t.is_pinned()) && t.is_contiguous() &&
           (int64_t)t.nbytes() > COPY_CHUNK && !t.requires_grad();
}

Tensor upload(const Tensor &host, c10::DeviceIndex index) {
    if (!copies_in_chunks(host, false)) return {};
    const c10::Device device(c10::DeviceType::CUDA, index);
    c10::DeviceGuard guard(device);
    at::AutoDispatchBelowADInplaceOrView no_views;
    Staging s(device);
    Tensor out = at::empty(host.sizes(), host.options().device(device));
    const Tensor from = as_bytes(host), to = as_bytes(out);
    const int64_t n = from.numel();
    for (int64_t at = 0, i = 0; at < n; at += COPY_CHUNK, i++) {
        const int64_t len = std::min(COPY_CHUNK, n - at);
        const Tensor pinned = s.buffer[i & 1].narrow(0, 0, len);
        if (i >= 2) s.done[i & 1].synchronize();         // the buffer's last chunk has left it
        pinned.copy_(from.narrow(0, at, len));
        to.narrow(0, at, len).copy_(pinned, true);
        s.done[i & 1].record(s.stream);
    }
    for (int64_t i = 0; i < std::min<int64_t>(2, (n + COPY_CHUNK - 1) / COPY_CHUNK); i++) s.done[i].synchronize();
    return out;
}

Tensor download(const Tensor &dev) {
    if (!copies_in_chunks(dev, true)) return {};
    c10::DeviceGuard guard(dev.device());
    at::AutoDispatchBelowADInplaceOrView no_views;
    Staging s(dev.device());
    Tensor out = at::empty(dev.sizes(), dev.options().device(c10::kCPU));
    const Tensor from = as_bytes(dev), to = as_bytes(out);
    const int64_t n = from.numel(), chunks = (n + COPY_CHUNK - 1) / COPY_CHUNK;
    auto length = [&](int64_t i) { return std::min(COPY_CHUNK, n - i * COPY_CHUNK); };
    for (int64_t i = 0; i <= chunks; i++) {
        if (i < chunks) {
            s.buffer[i & 1].narrow(0, 0, length(i)).copy_(from.narrow(0, i * COPY_CHUNK, length(i)), true);
            s.done[i & 1].record(s.stream);
        }
        if (i == 0) continue;
        s.done[(i - 1) & 1].synchronize();               // chunk i - 1 has arrived, chunk i is on its way
        to.narrow(0, (i - 1) * COPY_CHUNK, length(i - 1)).copy_(s.buffer[(i - 1) & 1].narrow(0, 0, length(i - 1)));
    }
    return out;
}

// ------------------------------------------------------------------ CPython side

// Arguments by position.  A tensor argument is a torch.Tensor or a Parameter (subclass): anything else, and a value
// of the wrong kind, raises TypeError.
struct Args {
    PyObject *const *a;
    Py_ssize_t n;
    const Tensor &tensor(Py_ssize_t i) const {
        if (!THPVariable_Check(a[i])) throw std::invalid_argument("a tensor is expected");
        return THPVariable_Unpack(a[i]);
    }
    Tensor optional(Py_ssize_t i) const { return a[i] == Py_None ? Tensor() : tensor(i); }
    int64_t integer(Py_ssize_t i) const {
        const long long v = PyLong_AsLongLong(a[i]);
        if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); throw std::invalid_argument("an integer is expected"); }
        return v;
    }
    bool truth(Py_ssize_t i) const { return PyObject_IsTrue(a[i]) == 1; }
};

// Runs fn (returning a Tensor) without the GIL and wraps the result, None for an undefined one.
template <typename Fn> PyObject *answer(const char *name, Py_ssize_t got, Py_ssize_t want, Fn &&fn) {
    HANDLE_TH_ERRORS
    if (got != want) {
        PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, want, got);
        return nullptr;
    }
    try {
        Tensor y = fn();
        if (!y.defined()) Py_RETURN_NONE;
        return THPVariable_Wrap(std::move(y));
    } catch (const std::invalid_argument &e) {
        PyErr_Format(PyExc_TypeError, "%s: %s", name, e.what());
    } catch (const Failed &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
    END_HANDLE_TH_ERRORS
}

struct NoGil {
    PyThreadState *state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

PyObject *py_bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 1 || !PyDict_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "bind takes a dict of function addresses");
        return nullptr;
    }
#define BIND(name)                                                                                 \
    do {                                                                                           \
        PyObject *v = PyDict_GetItemString(args[0], "lowbit_" #name);                              \
        void *p = v ? PyLong_AsVoidPtr(v) : nullptr;                                               \
        if (!p) {                                                                                  \
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, "lowbit_" #name);               \
            return nullptr;                                                                        \
        }                                                                                          \
        api.name = (decltype(api.name))p;                                                          \
    } while (0)
    BIND(last_error); BIND(blob_bytes); BIND(tileable); BIND(linear_scratch_bytes); BIND(linear);
    BIND(gated_mlp); BIND(dequantize_rows); BIND(dequantize); BIND(backward_ws); BIND(backward_workspace_bytes); BIND(backward_ws_applies); BIND(experts_workspace_bytes); BIND(experts_forward);
#undef BIND
    Py_RETURN_NONE;
}

// product(x [M, K] contiguous, w, qtype, layout, N) -> [M, N] in x's dtype; the caller has checked the arguments
PyObject *py_product(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return answer("product", n, 5, [&] {
        const Args a{args, n};
        const Tensor &x = a.tensor(0), &w = a.tensor(1);
        const int qtype = (int)a.integer(2), layout = (int)a.integer(3);
        const int64_t N = a.integer(4), M = x.size(0), K = x.size(1);
        NoGil free;
        return product(x, w, Tensor(), qtype, layout, M, N, K, {M, N});
    });
}

// linear(x, weight, bias or None, qtype, out_len, conver_to_half) -> y or None
PyObject *py_linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return answer("linear", n, 6, [&] {
        const Args a{args, n};
        const Tensor &x = a.tensor(0), &w = a.tensor(1);
        const Tensor bias = a.optional(2);
        const int qtype = (int)a.integer(3);
        const int64_t N = a.integer(4);
        const bool half = a.truth(5);
        NoGil free;
        return linear(x, w, bias, qtype, N, half);
    });
}

// linear_train(x, weight, bias or None, qtype, out_len) -> y or None
PyObject *py_linear_train(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return answer("linear_train", n, 5, [&] {
        const Args a{args, n};
        const Tensor &x = a.tensor(0), &w = a.tensor(1);
        const Tensor bias = a.optional(2);
        const int qtype = (int)a.integer(3);
        const int64_t N = a.integer(4);
        NoGil free;
        return linear_train(x, w, bias, qtype, N);
    });
}

// gated(x, w_gate, w_up, qtype, out_len, act) -> y or None
PyObject *py_gated(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return answer("gated", n, 6, [&] {
        const Args a{args, n};
        const Tensor &x = a.tensor(0), &wg = a.tensor(1), &wu = a.tensor(2);
        const int qtype = (int)a.integer(3), act = (int)a.integer(5);
        const int64_t N = a.integer(4);
        NoGil free;
        return gated(x, wg, wu, qtype, N, act);
    });
}

// embedding(ids, weight, qtype, num_embeddings, embedding_dim, tensor of the result's dtype) -> rows or None
PyObject *py_embedding(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return answer("embedding", n, 6, [&] {
        const Args a{args, n};
        const Tensor &ids = a.tensor(0), &w = a.tensor(1);
        const int qtype = (int)a.integer(2);
        const int64_t N = a.integer(3), K = a.integer(4);
        const at::ScalarType dtype = a.tensor(5).scalar_type();
        NoGil free;
        return embedding(ids, w, qtype, N, K, dtype);
    });
}

// experts(x, ids, weights, gates, ups, downs, qtype, hidden, inter, act) -> y or None
PyObject *py_experts(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return answer("experts", n, 10, [&] {
        const Args a{args, n};
        const Tensor &x = a.tensor(0), &ids = a.tensor(1), &weight = a.tensor(2), &g = a.tensor(3), &u = a.tensor(4), &d = a.tensor(5);
        const int qtype = (int)a.integer(6), act = (int)a.integer(9);
        const int64_t hidden = a.integer(7), inter = a.integer(8);
        NoGil free;
        return experts(x, ids, weight, g, u, d, qtype, hidden, inter, act);
    });
}

// upload(host tensor, device index) -> the tensor on that GPU, or None; complete when it returns
PyObject *py_upload(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return answer("upload", n, 2, [&] {
        const Args a{args, n};
        const Tensor &t = a.tensor(0);
        const auto index = (c10::DeviceIndex)a.integer(1);
        NoGil free;
        return upload(t, index);
    });
}

// download(tensor on a GPU) -> the tensor in host memory, or None
PyObject *py_download(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return answer("download", n, 1, [&] {
        const Args a{args, n};
        const Tensor &t = a.tensor(0);
        NoGil free;
        return download(t);
    });
}

// holds(parameter dicts, addresses): whether every dict's "weight" is a tensor whose data lies at the address (bytes of
// unsigned 64-bit numbers).  What ExpertWeights.check asks of each expert, 180 times for 60 experts: 0.3 us each in Python.
PyObject *py_holds(PyObject *, PyObject *const *args, Py_ssize_t n) {
    static PyObject *const weight = PyUnicode_InternFromString("weight");
    if (n != 2 || !PyTuple_Check(args[0]) || !PyBytes_Check(args[1]) ||
        PyBytes_GET_SIZE(args[1]) != PyTuple_GET_SIZE(args[0]) * (Py_ssize_t)sizeof(uint64_t)) {
        PyErr_SetString(PyExc_TypeError, "holds takes a tuple of dicts and as many addresses");
        return nullptr;
    }
    const uint64_t *want = (const uint64_t *)PyBytes_AS_STRING(args[1]);
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[0]); i++) {
        PyObject *d = PyTuple_GET_ITEM(args[0], i);
        PyObject *w = PyDict_Check(d) ? PyDict_GetItem(d, weight) : nullptr;
        if (!w || !THPVariable_Check(w)) Py_RETURN_FALSE;
        const Tensor &t = THPVariable_Unpack(w);
        if (!t.has_storage() || (uint64_t)(uintptr_t)t.const_data_ptr() != want[i]) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(bind), METHOD(product), METHOD(linear), METHOD(linear_train), METHOD(gated), METHOD(embedding), METHOD(experts), METHOD(upload),
                         METHOD(download), METHOD(holds),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "lowbit_torch", "native host path of the low-bit layers", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_lowbit_torch(void) { return PyModule_Create(&module); }
