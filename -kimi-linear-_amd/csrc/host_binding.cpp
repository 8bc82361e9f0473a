// The inference calls of the wrapper in native code: argument checks, output
// allocation (torch's caching allocator) and the C ABI call of kda_chunkwise,
// kda_recurrent and their gated and fused forms, and of the layer's
// pre-processing and output kernels.
//
// Each function takes the common form of its call -- HIP tensors of the types
// and layouts the kernels read as they are, nothing to differentiate, no
// dispatch mode or tensor subclass at work -- and returns None for any other
// call, before doing anything: the Python wrapper then takes its general path,
// which converts, copies or raises.  So a call has one meaning, and this file
// only answers for the part of it that needs no decision.  A launch that fails
// raises: it may have run.
//
// In Python a call's checks, its argument structure and its device and stream
// lookups took about 20 us (a decode step at B=1 takes 4 us on the GPU).
#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/extension.h>

#include <array>
#include <cmath>
#include <cstdint>
#include <optional>
#include <string>
#include <vector>

#include "kda_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

struct Fns {
    decltype(&kda_chunkwise_fwd) chunkwise = nullptr;
    decltype(&kda_recurrent_fwd) recurrent = nullptr;
    decltype(&kda_chunkwise_gated_fwd) chunkwise_gated = nullptr;
    decltype(&kda_recurrent_gated_fwd) recurrent_gated = nullptr;
    decltype(&kda_chunkwise_fused_fwd) fused = nullptr;
    decltype(&kda_chunkwise_long_fwd) long_fwd = nullptr;
    decltype(&kda_chunkwise_long_workspace_size) long_ws = nullptr;
    decltype(&kda_chunkwise_split_fwd) split_fwd = nullptr;
    decltype(&kda_chunkwise_split_workspace_size) split_ws = nullptr;
    decltype(&kda_prep_fwd) prep = nullptr;
    decltype(&kda_output_fwd) output = nullptr;
    decltype(&kda_linear_fwd) linear = nullptr;
    decltype(&kda_linear_wgrad) wgrad = nullptr;
    decltype(&kda_linear_wgrad_workspace_size) wgrad_ws = nullptr;
    decltype(&kda_status_str) status_str = nullptr;
};
Fns fn;
// torch._C._cuda_getCurrentRawStream and the wrapper's KdaError; kept for the process's life
PyObject* raw_stream = nullptr;
PyObject* error = nullptr;
at::DeviceType device_type = at::kCUDA;      // whose tensors the calls take

template <typename F>
void take(F& f, const py::dict& addr, const char* name) {
    f = reinterpret_cast<F>(addr[name].cast<uintptr_t>());
}

// The loaded library's entry points (name -> address), torch's stream lookup,
// the wrapper's exception and the type of the library's device.
void bind(const py::dict& addr, const py::object& stream_fn, const py::object& error_class, const std::string& device) {
    take(fn.chunkwise, addr, "kda_chunkwise_fwd");
    take(fn.recurrent, addr, "kda_recurrent_fwd");
    take(fn.chunkwise_gated, addr, "kda_chunkwise_gated_fwd");
    take(fn.recurrent_gated, addr, "kda_recurrent_gated_fwd");
    take(fn.fused, addr, "kda_chunkwise_fused_fwd");
    take(fn.long_fwd, addr, "kda_chunkwise_long_fwd");
    take(fn.long_ws, addr, "kda_chunkwise_long_workspace_size");
    take(fn.split_fwd, addr, "kda_chunkwise_split_fwd");
    take(fn.split_ws, addr, "kda_chunkwise_split_workspace_size");
    take(fn.prep, addr, "kda_prep_fwd");
    take(fn.output, addr, "kda_output_fwd");
    take(fn.linear, addr, "kda_linear_fwd");
    take(fn.wgrad, addr, "kda_linear_wgrad");
    take(fn.wgrad_ws, addr, "kda_linear_wgrad_workspace_size");
    take(fn.status_str, addr, "kda_status_str");
    device_type = at::Device(device).type();
    raw_stream = stream_fn.inc_ref().ptr();
    error = error_class.inc_ref().ptr();
}

// Whether the library refused the call, before any launch: the general path
// reports or answers it.  A failed launch is no refusal (the status is read
// after the launch and may be an older error of the thread: the kernels, or the
// first ones of several, may have run).  The general path would run them a
// second time, on a state updated in place, so it raises here.
bool refused(int status, const char* name) {
    if (status == KDA_ERR_LAUNCH) {
        PyErr_Format(error, "%s failed: %s", name, fn.status_str(status));
        throw py::error_already_set();
    }
    return status != KDA_OK;
}

int code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return KDA_DTYPE_F32;
        case at::kHalf: return KDA_DTYPE_F16;
        case at::kBFloat16: return KDA_DTYPE_BF16;
        default: return -1;
    }
}

// Whether nothing but the plain device tensors of one device takes part:
// checked per call, tensor by tensor.
struct Plain {
    at::Device dev;
    bool grad = at::GradMode::is_enabled();
    bool ok = true;
    explicit Plain(const Tensor& first)
        : dev(first.defined() ? first.device() : at::Device(at::kCPU)) {
        ok = dev.type() == device_type && c10::impl::TorchDispatchModeTLS::stack_len() == 0;
        add(first);
    }
    Plain& add(const Tensor& t) {
        static const c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                  c10::DispatchKey::FuncTorchGradWrapper,
                                                  c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor,
                                                  c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
        ok = ok && t.defined() && t.device() == dev && t.layout() == at::kStrided && !t.key_set().has_any(special) &&
             !(grad && t.requires_grad()) && !t._fw_grad(0).defined();
        return *this;
    }
    Plain& add(const OptTensor& t) {
        if (t) add(*t);
        return *this;
    }
};

void* stream_of(const at::Device& dev) {
    const py::int_ index(static_cast<int>(dev.index()));
    py::object s = py::reinterpret_steal<py::object>(PyObject_CallOneArg(raw_stream, index.ptr()));
    if (!s) throw py::error_already_set();
    return reinterpret_cast<void*>(s.cast<uintptr_t>());
}

// The interpreter lock given up for a scope (without the bookkeeping of
// py::gil_scoped_release, which a decode step's call of 6 us would notice).
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
    Unlocked() = default;
    Unlocked(const Unlocked&) = delete;
    Unlocked& operator=(const Unlocked&) = delete;
};

// f(stream), f the allocations and the C ABI call of one entry, on dev and its
// current stream.  Without the interpreter lock: an allocation or a launch into
// a full queue waits for the device, and other threads run meanwhile.
template <typename F>
int run(const at::Device& dev, F&& f) {
    void* stream = stream_of(dev);
    const Unlocked unlocked;
    const c10::DeviceGuard guard(dev);
    return f(stream);
}

bool sized(const Tensor& t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s); }

// [B, T, H, D]: contiguous channels, token rows that do not overlap.
bool rows_ok(const Tensor& t, int64_t D) {
    return (D == 1 || t.stride(3) == 1) && (t.size(1) <= 1 || t.stride(1) >= D);
}

void strides3(int64_t (&out)[3], const Tensor& t) {
    for (int i = 0; i < 3; ++i) out[i] = t.stride(i);
}

// From a tensor's first byte to past its last, the gaps of its strides included.
size_t extent(const Tensor& t) {
    int64_t last = 0;
    for (int64_t i = 0; i < t.dim(); ++i) last += (t.size(i) - 1) * t.stride(i);
    return t.numel() == 0 ? 0 : static_cast<size_t>((last + 1) * t.element_size());
}

bool overlaps(const Tensor& a, const Tensor& b) {
    const auto a0 = reinterpret_cast<uintptr_t>(a.data_ptr()), b0 = reinterpret_cast<uintptr_t>(b.data_ptr());
    return a0 < b0 + extent(b) && b0 < a0 + extent(a);
}

// kda_chunkwise / kda_recurrent (recurrent), with the gates' parameters their
// gated forms, with og also kda_chunkwise_fused.  segments > 1: the split of a
// long sequence the wrapper's rule asks for; transitions_first: in
// kda_chunkwise_split_fwd where that has a form.  (o, state) or None.
py::object core(bool recurrent, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& beta,
                const OptTensor& state, int64_t chunk_size, const std::optional<at::ScalarType>& state_dtype,
                const OptTensor& state_out, const OptTensor& a_log, const OptTensor& dt_bias, const OptTensor& og,
                const OptTensor& weight, double eps, int64_t segments, bool transitions_first) {
    Plain plain(q);
    plain.add(k).add(v).add(g).add(beta).add(state).add(state_out).add(a_log).add(dt_bias).add(og);
    if (!plain.ok || (weight && !weight->defined())) return py::none();
    if (q.dim() != 4 || v.dim() != 4) return py::none();
    const int64_t B = q.size(0), T = q.size(1), H = q.size(2), K = q.size(3), V = v.size(3);
    if (B * H == 0 || K <= 0 || V <= 0 || !sized(k, {B, T, H, K}) || !sized(g, {B, T, H, K}) ||
        !sized(v, {B, T, H, V}) || !sized(beta, {B, T, H}))
        return py::none();
    if (!recurrent && (chunk_size <= 0 || T % chunk_size != 0)) return py::none();
    const int dt = code(v), gt = code(g), bt = code(beta);
    if (dt < 0 || gt < 0 || bt < 0 || q.scalar_type() != v.scalar_type() || k.scalar_type() != v.scalar_type())
        return py::none();
    const bool gated = a_log.has_value();
    if (!recurrent) {
        if (!gated && (gt != KDA_DTYPE_F32 || bt != KDA_DTYPE_F32)) return py::none();
        if (gated && dt != KDA_DTYPE_F32 && (gt != dt || bt != dt)) return py::none();
    }
    if (!rows_ok(q, K) || !rows_ok(k, K) || !rows_ok(g, K) || !rows_ok(v, V) || (T > 1 && beta.stride(1) < 1))
        return py::none();
    if (gated != dt_bias.has_value()) return py::none();
    if (gated && (a_log->scalar_type() != at::kFloat || dt_bias->scalar_type() != at::kFloat ||
                  a_log->numel() != H * K || dt_bias->numel() != H * K || !a_log->is_contiguous() ||
                  !dt_bias->is_contiguous()))
        return py::none();
    const at::ScalarType st = state_dtype ? *state_dtype : v.scalar_type();
    if (st != at::kFloat && st != at::kHalf && st != at::kBFloat16) return py::none();
    if (state && (!sized(*state, {B, H, K, V}) || code(*state) < 0 || !state->is_contiguous())) return py::none();
    if (state_out) {
        if (!sized(*state_out, {B, H, K, V}) || !state_out->is_contiguous() || state_out->scalar_type() != st ||
            state_out->requires_grad())
            return py::none();
        if (state && overlaps(*state, *state_out) &&
            !(recurrent && state->data_ptr() == state_out->data_ptr() && state->scalar_type() == st))
            return py::none();
    }
    if (og) {
        if (recurrent || !weight || dt == KDA_DTYPE_F32 || (K != 64 && K != 128) || (V != 64 && V != 128) ||
            !sized(*og, {B, T, H * V}) || og->scalar_type() != v.scalar_type() || og->stride(2) != 1 ||
            (T > 1 && og->stride(1) < H * V) || weight->device() != plain.dev || weight->numel() != H * V)
            return py::none();
    }
    if (segments > 1) {
        if (recurrent || gated || og || state_out) return py::none();
        // one batch stride must serve the split views (sequences back to back)
        for (const Tensor* x : {&q, &k, &v, &g, &beta})
            if (B != 1 && x->stride(0) != T * x->stride(1)) segments = 1;
    }

    Tensor o, s, keep;                               // keep: alive until the launches that read it are enqueued
    const int status = run(plain.dev, [&](void* stream) -> int {
        o = at::empty({B, T, H, V}, v.options().requires_grad(false));
        s = state_out ? *state_out : at::empty({B, H, K, V}, v.options().dtype(st).requires_grad(false));
        kda_fwd_args a{};
        a.B = B; a.T = T; a.H = H; a.K = K; a.V = V;
        a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.g = g.data_ptr(); a.beta = beta.data_ptr();
        strides3(a.q_stride, q);
        strides3(a.k_stride, k);
        strides3(a.v_stride, v);
        strides3(a.g_stride, g);
        strides3(a.beta_stride, beta);
        a.qkv_dtype = dt; a.g_dtype = gt; a.beta_dtype = bt;
        a.state_in = state ? state->data_ptr() : nullptr;
        a.state_in_dtype = state ? code(*state) : KDA_DTYPE_F32;
        a.state_out = s.data_ptr();
        a.state_out_dtype = code(s);
        a.o = o.data_ptr();
        a.scale = static_cast<float>(std::pow(static_cast<double>(K), -0.5));
        a.clamp_fp16_out = recurrent ? 1 : 0;
        a.chunk_size = recurrent ? 1 : chunk_size;
        kda_gate_args ga{};
        if (gated) {
            ga.a_log = static_cast<const float*>(a_log->data_ptr());
            ga.dt_bias = static_cast<const float*>(dt_bias->data_ptr());
        }
        if (segments > 1) {
            // the form whose transition columns end when they are zero, where there is one
            const size_t split = transitions_first ? fn.split_ws(B, T, H, K, V, segments) : 0;
            const size_t bytes = split != 0 ? split : fn.long_ws(B, T, H, K, V, segments);
            keep = at::empty({static_cast<int64_t>(bytes)}, v.options().dtype(at::kByte).requires_grad(false));
            return (split != 0 ? fn.split_fwd : fn.long_fwd)(&a, segments, keep.data_ptr(), stream);
        }
        if (og) {
            keep = weight->detach().to(at::kFloat).contiguous();
            kda_out_epilogue e{};
            e.gate = og->data_ptr();
            e.gate_stride[0] = og->stride(0);
            e.gate_stride[1] = og->stride(1);
            e.weight = static_cast<const float*>(keep.data_ptr());
            e.eps = static_cast<float>(eps);
            return fn.fused(&a, gated ? &ga : nullptr, &e, stream);
        }
        if (gated) return (recurrent ? fn.recurrent_gated : fn.chunkwise_gated)(&a, &ga, stream);
        return (recurrent ? fn.recurrent : fn.chunkwise)(&a, stream);
    });
    if (refused(status, recurrent ? "kda_recurrent" : "kda_chunkwise")) return py::none();
    return py::make_tuple(o, s);
}

// Vector accesses of n elements: base and row strides aligned to them.
bool vec_ok(const Tensor& t, int64_t n) {
    if (reinterpret_cast<uintptr_t>(t.data_ptr()) % (n * t.element_size()) != 0) return false;
    for (int64_t i = 0; i + 1 < t.dim(); ++i)
        if (t.stride(i) % n != 0) return false;
    return true;
}

// kda_prep: (q, k, v, g or None, beta or None, (hq, hk, hv) or None) or None.
py::object prep(const std::array<Tensor, 3>& x, const std::array<Tensor, 3>& w, const std::array<OptTensor, 3>& bias,
                const OptTensor& gk, const OptTensor& a_log, const OptTensor& dt_bias, const OptTensor& beta_logit,
                int64_t H, int64_t K, int64_t V, double l2_eps, const std::array<OptTensor, 3>& hist,
                const std::array<OptTensor, 3>& hist_out, bool want_hist) {
    Plain plain(x[0]);
    for (int i = 0; i < 3; ++i) plain.add(x[i]).add(w[i]).add(bias[i]).add(hist[i]).add(hist_out[i]);
    const bool gates = gk.has_value();
    if (gates) plain.add(gk).add(a_log).add(dt_bias).add(beta_logit);
    if (!plain.ok || x[0].dim() != 3 || H <= 0 || (K != 64 && K != 128 && K != 256) ||
        (V != 64 && V != 128 && V != 256))
        return py::none();
    const int64_t B = x[0].size(0), T = x[0].size(1);
    const int dt = code(x[0]), wt = code(w[0]);
    if (B == 0 || T == 0 || dt < 0 || wt < 0 || w[0].dim() != 3) return py::none();
    const int64_t cs = w[0].size(2), keep = cs - 1;
    if (cs < 1 || cs > 4) return py::none();
    const bool have_out = hist_out[0].has_value();
    if (have_out && want_hist) return py::none();
    for (int i = 0; i < 3; ++i) {
        const int64_t Dh = i == 2 ? V : K, D = H * Dh;
        if (!sized(x[i], {B, T, D}) || x[i].scalar_type() != x[0].scalar_type() || x[i].stride(2) != 1 ||
            !vec_ok(x[i], Dh / 64) || !sized(w[i], {D, 1, cs}) || code(w[i]) != wt || !w[i].is_contiguous())
            return py::none();
        if (bias[i] && (!sized(*bias[i], {D}) || code(*bias[i]) != wt || !bias[i]->is_contiguous())) return py::none();
        for (const OptTensor* h : {&hist[i], &hist_out[i]})
            if (*h && (!sized(**h, {B, keep, D}) || (**h).scalar_type() != x[0].scalar_type() ||
                       !(**h).is_contiguous()))
                return py::none();
        if (hist[i].has_value() != hist[0].has_value() || hist_out[i].has_value() != have_out) return py::none();
    }
    if (gates) {
        if (!a_log || !dt_bias || !beta_logit || !sized(*gk, {B, T, H * K}) || gk->stride(2) != 1 ||
            gk->scalar_type() != x[0].scalar_type() || !vec_ok(*gk, K / 64) || !sized(*beta_logit, {B, T, H}) ||
            (H > 1 && beta_logit->stride(2) != 1) || beta_logit->scalar_type() != x[0].scalar_type() ||
            a_log->numel() != H * K || dt_bias->numel() != H * K || code(*a_log) < 0 ||
            a_log->scalar_type() != dt_bias->scalar_type() || !a_log->is_contiguous() || !dt_bias->is_contiguous())
            return py::none();
    }

    Tensor out[3], g, beta, hn[3];
    const int status = run(plain.dev, [&](void* stream) -> int {
        const auto opt = x[0].options().requires_grad(false);
        for (int i = 0; i < 3; ++i) out[i] = at::empty({B, T, H, i == 2 ? V : K}, opt);
        kda_prep_args a{};
        a.B = B; a.T = T; a.H = H; a.K = K; a.V = V; a.conv_size = cs;
        for (int i = 0; i < 3; ++i) {
            a.x[i] = x[i].data_ptr();
            a.x_stride[i][0] = x[i].stride(0);
            a.x_stride[i][1] = x[i].stride(1);
            a.conv_w[i] = w[i].data_ptr();
            a.conv_b[i] = bias[i] ? bias[i]->data_ptr() : nullptr;
            a.hist_in[i] = hist[i] ? hist[i]->data_ptr() : nullptr;
            if (want_hist) hn[i] = at::empty({B, keep, H * (i == 2 ? V : K)}, opt);
            else if (have_out) hn[i] = *hist_out[i];
            a.hist_out[i] = hn[i].defined() ? hn[i].data_ptr() : nullptr;
        }
        a.w_dtype = wt;
        a.p_dtype = KDA_DTYPE_F32;
        if (gates) {
            g = at::empty({B, T, H, K}, opt.dtype(at::kFloat));
            beta = at::empty({B, T, H}, opt.dtype(at::kFloat));
            a.gk = gk->data_ptr();
            a.gk_stride[0] = gk->stride(0);
            a.gk_stride[1] = gk->stride(1);
            a.a_log = a_log->data_ptr();
            a.dt_bias = dt_bias->data_ptr();
            a.p_dtype = code(*a_log);
            a.beta_logit = beta_logit->data_ptr();
            a.beta_stride[0] = beta_logit->stride(0);
            a.beta_stride[1] = beta_logit->stride(1);
            a.g = static_cast<float*>(g.data_ptr());
            a.beta = static_cast<float*>(beta.data_ptr());
        }
        a.q = out[0].data_ptr();
        a.k = out[1].data_ptr();
        a.v = out[2].data_ptr();
        a.l2_eps = static_cast<float>(l2_eps);
        a.x_dtype = dt;
        return fn.prep(&a, stream);
    });
    if (refused(status, "kda_prep_fwd")) return py::none();
    py::object pg = py::none(), pb = py::none(), ph = py::none();
    if (gates) pg = py::cast(g), pb = py::cast(beta);
    if (hn[0].defined()) ph = py::make_tuple(hn[0], hn[1], hn[2]);
    return py::make_tuple(out[0], out[1], out[2], pg, pb, ph);
}

// kda_output: y [B, T, H V] or None.
py::object output(const Tensor& o, const Tensor& gate, const Tensor& weight, double eps) {
    Plain plain(o);
    plain.add(gate).add(weight);
    if (!plain.ok || o.dim() != 4 || o.numel() == 0) return py::none();
    const int64_t B = o.size(0), T = o.size(1), H = o.size(2), V = o.size(3);
    if ((V != 64 && V != 128 && V != 256) || code(o) < 0 || code(weight) < 0 || o.stride(3) != 1 ||
        !sized(gate, {B, T, H * V}) || gate.scalar_type() != o.scalar_type() || gate.stride(2) != 1 ||
        !sized(weight, {H, V}) || !weight.is_contiguous() || !vec_ok(o, V / 64) || !vec_ok(gate, V / 64))
        return py::none();
    Tensor y;
    const int status = run(plain.dev, [&](void* stream) -> int {
        y = at::empty({B, T, H * V}, o.options().requires_grad(false));
        kda_output_args a{};
        a.B = B; a.T = T; a.H = H; a.V = V;
        a.o = o.data_ptr();
        strides3(a.o_stride, o);
        a.gate = gate.data_ptr();
        a.gate_stride[0] = gate.stride(0);
        a.gate_stride[1] = gate.stride(1);
        a.weight = weight.data_ptr();
        a.w_dtype = code(weight);
        a.y = y.data_ptr();
        a.eps = static_cast<float>(eps);
        a.x_dtype = code(o);
        return fn.output(&a, stream);
    });
    if (refused(status, "kda_output_fwd")) return py::none();
    return py::cast(y);
}

// Rows of x [B, T, K] one stride apart, as few as kda_linear_fwd takes, and w [N, K].
bool linear_ok(const Plain& plain, const Tensor& x, const Tensor& w) {
    const auto dt = x.scalar_type();
    return plain.ok && (dt == at::kHalf || dt == at::kBFloat16) && x.dim() == 3 && x.numel() > 0 && w.numel() > 0 &&
           w.dim() == 2 && x.size(0) <= 64 && x.size(1) <= 64 && x.size(0) * x.size(1) <= 64 && x.stride(2) == 1 &&
           (x.size(0) == 1 || x.size(1) == 1 || x.stride(0) == x.size(1) * x.stride(1)) && w.size(1) == x.size(2) &&
           w.scalar_type() == dt && w.is_contiguous();
}

int64_t row_stride(const Tensor& x) { return x.size(1) == 1 ? x.stride(0) : x.stride(1); }

void linear_operands(kda_linear_args& a, int i, const Tensor& x, const Tensor& w, const Tensor& y) {
    a.x[i] = x.data_ptr();
    a.x_stride[i] = row_stride(x);
    a.w[i] = w.data_ptr();
    a.N[i] = w.size(0);
    a.y[i] = y.data_ptr();
}

// Autocast would choose the projection's type: its calls are the general path's.
bool autocast_on() { return at::autocast::is_autocast_enabled(at::kCUDA); }

// x w^T of few rows, [B, T, N]; residual [B, T, N]: their sum; out: written
// there.  The result, or None for the calls of the library product.
py::object linear(const Tensor& x, const Tensor& w, const OptTensor& residual, const OptTensor& out) {
    Plain plain(x);
    plain.add(w).add(residual).add(out);
    if (!linear_ok(plain, x, w) || autocast_on()) return py::none();
    const int64_t B = x.size(0), T = x.size(1), N = w.size(0);
    if (residual && (!sized(*residual, {B, T, N}) || residual->scalar_type() != x.scalar_type() ||
                     residual->stride(2) != 1 ||
                     (B > 1 && T > 1 && residual->stride(0) != T * residual->stride(1))))
        return py::none();
    if (out && (!sized(*out, {B, T, N}) || out->scalar_type() != x.scalar_type() || !out->is_contiguous() ||
                overlaps(*out, x) || overlaps(*out, w) || (residual && overlaps(*out, *residual))))
        return py::none();
    Tensor y;
    const int status = run(plain.dev, [&](void* stream) -> int {
        y = out ? *out : at::empty({B, T, N}, x.options().requires_grad(false));
        kda_linear_args a{};
        a.M = B * T;
        a.K = x.size(2);
        linear_operands(a, 0, x, w, y);
        if (residual) {
            a.residual = residual->data_ptr();
            a.residual_stride = row_stride(*residual);
        }
        a.dtype = code(x);
        return fn.linear(&a, stream);
    });
    if (refused(status, "kda_linear_fwd")) return py::none();
    return py::cast(y);
}

// Two such products of one depth in one launch: (y0, y1) or None.
py::object linear2(const Tensor& x0, const Tensor& w0, const Tensor& x1, const Tensor& w1) {
    Plain plain(x0);
    plain.add(w0).add(x1).add(w1);
    if (!linear_ok(plain, x0, w0) || !linear_ok(plain, x1, w1) || !x0.sizes().equals(x1.sizes()) ||
        x0.scalar_type() != x1.scalar_type() || autocast_on())
        return py::none();
    Tensor y0, y1;
    const int status = run(plain.dev, [&](void* stream) -> int {
        const auto opt = x0.options().requires_grad(false);
        y0 = at::empty({x0.size(0), x0.size(1), w0.size(0)}, opt);
        y1 = at::empty({x0.size(0), x0.size(1), w1.size(0)}, opt);
        kda_linear_args a{};
        a.M = x0.size(0) * x0.size(1);
        a.K = x0.size(2);
        linear_operands(a, 0, x0, w0, y0);
        linear_operands(a, 1, x1, w1, y1);
        a.dtype = code(x0);
        return fn.linear(&a, stream);
    });
    if (refused(status, "kda_linear_fwd")) return py::none();
    return py::make_tuple(y0, y1);
}

// Rows of [B, T, D] one stride apart.
bool one_stride(const Tensor& t) {
    return t.stride(2) == 1 && (t.size(0) == 1 || t.size(1) == 1 || t.stride(0) == t.size(1) * t.stride(1));
}

// dy^T x over the tokens, [N, K], or None for the calls of the library product.
py::object linear_wgrad(const Tensor& dy, const Tensor& x) {
    Plain plain(dy);
    plain.add(x);
    const auto dt = dy.scalar_type();
    if (!plain.ok || (dt != at::kHalf && dt != at::kBFloat16) || x.scalar_type() != dt || dy.dim() != 3 ||
        x.dim() != 3 || dy.size(0) != x.size(0) || dy.size(1) != x.size(1) || dy.numel() == 0 || x.numel() == 0 ||
        !one_stride(dy) || !one_stride(x))
        return py::none();
    kda_linear_wgrad_args a{};
    a.M = dy.size(0) * dy.size(1);
    a.N = dy.size(2);
    a.K = x.size(2);
    const size_t bytes = fn.wgrad_ws(a.M, a.N, a.K);
    if (bytes == 0) return py::none();
    Tensor dw;
    const int status = run(plain.dev, [&](void* stream) -> int {
        const auto opt = x.options().requires_grad(false);
        dw = at::empty({a.N, a.K}, opt);
        const Tensor ws = at::empty({static_cast<int64_t>(bytes)}, opt.dtype(at::kByte));
        a.dy = dy.data_ptr();
        a.dy_stride = row_stride(dy);
        a.x = x.data_ptr();
        a.x_stride = row_stride(x);
        a.dw = dw.data_ptr();
        a.workspace = ws.data_ptr();
        a.dtype = code(x);
        return fn.wgrad(&a, stream);
    });
    if (refused(status, "kda_linear_wgrad")) return py::none();
    return py::cast(dw);
}

// What decides whether a copy made of these parameters is still theirs:
// storage address, version, type and device of each.
py::bytes params_key(const std::vector<Tensor>& params) {
    std::string s;
    s.reserve(params.size() * 24);
    for (const Tensor& p : params) {
        const uint64_t w[3] = {reinterpret_cast<uint64_t>(p.data_ptr()), static_cast<uint64_t>(p._version()),
                               static_cast<uint64_t>(p.scalar_type()) << 32 |
                                   static_cast<uint64_t>(static_cast<uint8_t>(p.device().type())) << 8 |
                                   static_cast<uint64_t>(static_cast<uint8_t>(p.device().index()))};
        s.append(reinterpret_cast<const char*>(w), sizeof(w));
    }
    return py::bytes(s);
}

}  // namespace

PYBIND11_MODULE(_kda_host, m) {
    m.def("abi_version", [] { return KDA_ABI_VERSION; });
    m.attr("torch_version") = KDA_TORCH_VERSION;    // it was compiled against; its C++ interface is not stable
    m.def("bind", &bind);
    m.def("core", [](bool recurrent, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g,
                     const Tensor& beta, const OptTensor& state, int64_t chunk_size,
                     const std::optional<at::ScalarType>& state_dtype, const OptTensor& state_out,
                     const OptTensor& a_log, const OptTensor& dt_bias, const OptTensor& og, const OptTensor& weight,
                     double eps, int64_t segments) {
        return core(recurrent, q, k, v, g, beta, state, chunk_size, state_dtype, state_out, a_log, dt_bias, og, weight,
                    eps, segments, true);
    });
    m.def("core", &core);
    m.def("prep", &prep);
    m.def("output", &output);
    m.def("linear", &linear);
    m.def("linear2", &linear2);
    m.def("linear_wgrad", &linear_wgrad);
    m.def("params_key", &params_key);
}
