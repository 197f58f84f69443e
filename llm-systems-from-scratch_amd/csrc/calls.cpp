// The package's operators from Python in one native call each, for calls in the plain form.
//
// A call of a few microseconds of kernels cost 10 to 15 us of Python (checks, strides, allocations, ctypes), a small training call of one
// attention layer 145, part of it the autograd engine's thread waiting for the interpreter: here its backward is a C++ node that never
// asks for it.  Us of host time a call, ops.py alone / through this file: decode 11.0 / 4.8, packed prefill 16.4 / 5.1, router + experts +
// norm 38 / 20, rotation + cache write + portion over an fp8 cache 46 / 19, mixer + norm 28 / 16; forward and backward of a few short
// sequences 145 / 72.
//
// Every function here takes what its counterpart in ops.py takes, in a fixed order, and returns None when anything about the call
// is not plain (a tensor subclass, a mode of torch that wants to see operators, mixed devices, a layout that needs a copy, an argument that
// is wrong): ops.py then does it, with its checks and its errors.  So nothing is refused here, and what is accepted here is what
// ops.py would have handed to the same C function with the same arguments.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <atomic>
#include <cmath>
#include <optional>
#include <tuple>

#include "../../include/mi355_attn.h"

namespace {

using at::Tensor;
constexpr auto kBF16 = at::kBFloat16, kF32 = at::kFloat, kI32 = at::kInt, kI64 = at::kLong;

// ---- what makes a call plain --------------------------------------------------------------------
const c10::DispatchKeySet kOdd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                c10::DispatchKey::ZeroTensor});

struct Args {
    PyObject* const* at;
    bool ok;
    c10::Device device{c10::DeviceType::CPU};

    Args(PyObject* const* args, Py_ssize_t n, Py_ssize_t want) : at(args), ok(n == want) {}

    const Tensor* any(int i) {
        if (!ok || !THPVariable_CheckExact(at[i])) return fail();
        const Tensor& t = THPVariable_Unpack(at[i]);
        if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_nested() || t.key_set().has_any(kOdd)) return fail();
        if (device.is_cpu()) device = t.device();
        else if (t.device() != device) return fail();
        return &t;
    }
    const Tensor* tensor(int i, at::ScalarType dtype, int64_t dim) {
        const Tensor* t = any(i);
        return t && (t->scalar_type() != dtype || t->dim() != dim) ? fail() : t;
    }
    // contiguous, of the given type and sizes
    const Tensor* whole(int i, at::ScalarType dtype, at::IntArrayRef sizes) {
        const Tensor* t = any(i);
        return t && (t->scalar_type() != dtype || t->sizes() != sizes || !t->is_contiguous()) ? fail() : t;
    }
    // rows that may be strided
    const Tensor* matrix(int i, at::ScalarType dtype) {
        const Tensor* t = tensor(i, dtype, 2);
        return t && t->stride(1) != 1 && t->size(1) > 1 ? fail() : t;
    }
    // (tokens, heads, d_head) with contiguous heads, 16-byte aligned rows
    const Tensor* heads(int i, at::ScalarType dtype) {
        const Tensor* t = tensor(i, dtype, 3);
        return t && (t->stride(2) != 1 || t->stride(1) != t->size(2) || t->stride(0) % 8 || !aligned(*t)) ? fail() : t;
    }
    bool none(int i) const { return at[i] == Py_None; }
    bool flag(int i) {
        if (at[i] != Py_True && at[i] != Py_False) ok = false;
        return at[i] == Py_True;
    }
    int64_t integer(int i) {
        if (!ok || !PyLong_CheckExact(at[i])) return fail(), 0;
        int overflow = 0;
        const long long v = PyLong_AsLongLongAndOverflow(at[i], &overflow);
        if (overflow || v > 0x7fffffffLL || v < -0x7fffffffLL) ok = false;
        return v;
    }
    double number(int i) {
        if (PyFloat_CheckExact(at[i])) return PyFloat_AS_DOUBLE(at[i]);
        return (double)integer(i);
    }
    static bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
    void need(bool what) { ok = ok && what; }

    // nothing of torch's wants to see the operators (a trace records the Python functions' calls and would keep these results as
    // constants), and the tensors' GPU is the current one
    bool plain() const {
        const auto included = c10::impl::tls_local_dispatch_key_set().included_;
        return ok && device.is_cuda() && !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() &&
               !included.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !included.has(c10::DispatchKey::Tracer) &&
               c10::hip::current_device() == device.index();
    }

private:
    const Tensor* fail() {
        ok = false;
        return nullptr;
    }
};

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// The error that _lib.check raises
void check(int rc, const char* what) {
    if (rc == 0) return;
    const std::string msg = mi355_last_error();
    if (rc < 0) C10_THROW_ERROR(ValueError, std::string(what) + ": " + msg + " (code " + std::to_string(rc) + ")");
    C10_THROW_ERROR(Error, std::string(what) + ": HIP error " + std::to_string(rc) + ": " + msg);
}

void* stream_of(const c10::Device& d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }
Tensor make(at::IntArrayRef sizes, at::ScalarType dtype, const c10::Device& d) { return at::empty(sizes, at::TensorOptions().dtype(dtype).device(d)); }
const void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }
int64_t bytes(const Tensor& t) { return t.numel() * (int64_t)t.element_size(); }

int compute_units(const c10::Device& d) {
    static std::array<std::atomic<int>, 64> units{};
    const int i = d.index();
    if (i < 0 || i >= (int)units.size()) return 256;
    int n = units[i].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, i) != hipSuccess) n = 256;
        units[i].store(n, std::memory_order_relaxed);
    }
    return n;
}

// ---- attention over packed or dense tensors ----------------------------------------------------------
// Whether the rows of t are what the kernels read: 16 bytes at a time, strides of whole pieces
bool whole_rows(const Tensor& t) {
    bool good = t.stride(-1) == 1 && Args::aligned(t);
    for (int64_t i = 0; i + 1 < t.dim(); ++i) good = good && t.stride(i) % 8 == 0;
    return good;
}
Tensor rows16(const Tensor& t) { return whole_rows(t) ? t : t.contiguous(); }
struct Strides {                       // [batch, head, row]
    int64_t s[3];
    explicit Strides(const Tensor& t) {
        const bool packed = t.dim() == 3;
        s[0] = packed ? 0 : t.stride(0);
        s[1] = t.stride(1);
        s[2] = packed ? t.stride(0) : t.stride(2);
    }
    operator const int64_t*() const { return s; }
};

struct Shape {
    bool packed, causal;
    int B, Hq, Hkv, Sq, Sk, D;
    double scale;
    int mode() const { return causal ? MI355_MASK_CAUSAL : MI355_MASK_NONE; }
};

// out and the log-sum-exp of a forward pass for training
std::pair<Tensor, Tensor> forward_lse(const Tensor& q, const Tensor& k, const Tensor& v, const int32_t* cu_q, const int32_t* cu_k, const Shape& s) {
    const auto dev = q.device();
    const Tensor out = s.packed ? make(q.sizes(), kBF16, dev) : make({s.B, s.Sq, s.Hq, s.D}, kBF16, dev).permute({0, 2, 1, 3});
    const Tensor lse = s.packed ? make({s.Hq, q.size(0)}, kF32, dev) : make({s.B, s.Hq, s.Sq}, kF32, dev);
    const int64_t ls[2] = {s.packed ? 0 : lse.stride(0), s.packed ? lse.stride(0) : lse.stride(1)};
    check(mi355_prefill_fwd_lse(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), (float*)lse.data_ptr(), Strides(q), Strides(k), Strides(v),
                                Strides(out), ls, cu_q, cu_k, s.B, s.Hq, s.Hkv, s.Sq, s.Sk, s.D, (float)s.scale, s.mode(), MI355_BF16, stream_of(dev)),
          "mi355_prefill_fwd_lse");
    return {out, lse};
}

Tensor grad_like(const Tensor& t, at::ScalarType dtype) {
    Tensor g = at::empty_like(t, t.options().dtype(dtype));
    bool good = g.stride(-1) == 1;
    for (int64_t i = 0; i + 1 < g.dim(); ++i) good = good && g.stride(i) % 8 == 0;
    return good ? g : make(t.sizes(), dtype, t.device());
}

torch::autograd::variable_list backward_of(const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& out0, const Tensor& dout0, const Tensor& lse,
                                           const int32_t* cu_q, const int32_t* cu_k, const Shape& s, int f32) {
    const c10::DeviceGuard guard(q0.device());
    const auto dev = q0.device();
    const Tensor q = rows16(q0), k = rows16(k0), v = rows16(v0), out = rows16(out0), dout = rows16(dout0);
    const Tensor dq = grad_like(q, f32 & 1 ? kF32 : kBF16), dk = grad_like(k, f32 & 2 ? kF32 : kBF16), dv = grad_like(v, f32 & 4 ? kF32 : kBF16);
    const int64_t ls[2] = {s.packed ? 0 : lse.stride(0), s.packed ? lse.stride(0) : lse.stride(1)};
    const int64_t total_q = s.packed ? q.size(0) : 0, total_k = s.packed ? k.size(0) : 0;
    Tensor workspace;
    int64_t need = 0;
    if (std::max(s.Sq, s.Sk) > 64) {
        need = mi355_prefill_bwd_ds_workspace(s.B, s.Hq, s.Hkv, s.Sq, s.Sk, s.D, s.mode(), s.packed, !s.packed || cu_q == cu_k, total_q, total_k);
        if (need) {
            try {
                workspace = make({need + 4 * lse.numel()}, at::kByte, dev);
            } catch (const c10::OutOfMemoryError&) {       // (the other form needs none of it)
            }
        }
    }
    if (workspace.defined()) {
        char* ws = (char*)workspace.data_ptr();
        check(mi355_prefill_bwd_ds(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), dout.data_ptr(), (const float*)lse.data_ptr(), (float*)(ws + need),
                                   dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), Strides(q), Strides(k), Strides(v), Strides(out), Strides(dout), Strides(dq),
                                   Strides(dk), Strides(dv), ls, cu_q, cu_k, f32, s.B, s.Hq, s.Hkv, s.Sq, s.Sk, s.D, (float)s.scale, s.mode(), MI355_BF16,
                                   total_q, total_k, ws, need, stream_of(dev)),
              "mi355_prefill_bwd_ds");
    } else {
        const Tensor delta = at::empty_like(lse);
        const int64_t no_mask[3] = {0, 0, 0};
        check(mi355_prefill_bwd_typed(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), dout.data_ptr(), (const float*)lse.data_ptr(),
                                      (float*)delta.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), Strides(q), Strides(k), Strides(v), Strides(out),
                                      Strides(dout), Strides(dq), Strides(dk), Strides(dv), ls, cu_q, cu_k, nullptr, no_mask, f32, s.B, s.Hq, s.Hkv, s.Sq,
                                      s.Sk, s.D, (float)s.scale, s.mode(), MI355_BF16, stream_of(dev)),
              "mi355_prefill_bwd_typed");
    }
    return {dq, dk, dv};
}

int f32_bits(const Tensor& q, const Tensor& k, const Tensor& v) {
    return (q.scalar_type() == kF32 ? 1 : 0) | (k.scalar_type() == kF32 ? 2 : 0) | (v.scalar_type() == kF32 ? 4 : 0);
}

// q, k and v with what is fp32 among them rounded: in one launch where their elements fill their memory
std::array<Tensor, 3> bf16(const Tensor& q, const Tensor& k, const Tensor& v) {
    const Tensor* t[3] = {&q, &k, &v};
    std::array<Tensor, 3> r;
    const float* in[3] = {nullptr, nullptr, nullptr};
    void* out[3] = {nullptr, nullptr, nullptr};
    int64_t n[3] = {0, 0, 0};
    for (int i = 0; i < 3; ++i) {
        if (t[i]->scalar_type() == kBF16) {
            r[i] = *t[i];
        } else if (!t[i]->is_non_overlapping_and_dense() || !Args::aligned(*t[i]) || t[i]->numel() > 1LL << 32) {
            r[i] = t[i]->to(kBF16);
        } else {
            r[i] = at::empty_like(*t[i], t[i]->options().dtype(kBF16));
            in[i] = (const float*)t[i]->data_ptr();
            out[i] = r[i].data_ptr();
            n[i] = t[i]->numel();
        }
    }
    if (in[0] || in[1] || in[2]) check(mi355_round_operands(in, out, n, stream_of(q.device())), "mi355_round_operands");
    return r;
}

// forward_lse of short heads with fp32 among q, k and v, which it rounds: q, k, v become what the backward reads
bool forward_rounded(Tensor& q, Tensor& k, Tensor& v, const Shape& s, Tensor& out, Tensor& lse) {
    Tensor* t[3] = {&q, &k, &v};
    const int f32 = f32_bits(q, k, v);
    if (f32 == 0 || !((float)s.scale > 0.f) || !mi355_prefill_fwd_rounds(s.Hq, s.Hkv, s.Sq, s.Sk, s.D, s.mode())) return false;
    Tensor r[3];
    for (int i = 0; i < 3; ++i) {
        const int64_t row = t[i]->stride(2);               // (a conversion in front brings rows together that are further apart)
        if (!whole_rows(*t[i]) || row <= 0 || row >= (1 << 24)) return false;
        if (t[i]->scalar_type() != kF32) continue;
        r[i] = at::empty_like(*t[i], t[i]->options().dtype(kBF16));
        if (!whole_rows(r[i])) return false;
    }
    const auto dev = q.device();
    out = make({s.B, s.Sq, s.Hq, s.D}, kBF16, dev).permute({0, 2, 1, 3});
    lse = make({s.B, s.Hq, s.Sq}, kF32, dev);
    const int64_t ls[2] = {lse.stride(0), lse.stride(1)};
    void* to[3];
    for (int i = 0; i < 3; ++i) to[i] = r[i].defined() ? r[i].data_ptr() : nullptr;
    check(mi355_prefill_fwd_lse_rounded(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), (float*)lse.data_ptr(), Strides(q), Strides(k), Strides(v),
                                        Strides(out), ls, f32, to[0], to[1], to[2], Strides(r[0].defined() ? r[0] : q), Strides(r[1].defined() ? r[1] : k),
                                        Strides(r[2].defined() ? r[2] : v), s.B, s.Hq, s.Hkv, s.Sq, s.Sk, s.D, (float)s.scale, s.mode(), stream_of(dev)),
          "mi355_prefill_fwd_lse_rounded");
    for (int i = 0; i < 3; ++i)
        if (r[i].defined()) *t[i] = r[i];
    return true;
}

// The counterparts of _DensePrefillFn and _VarlenPrefillFn
struct DenseFn : torch::autograd::Function<DenseFn> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q0, const Tensor& k0, const Tensor& v0, bool causal, double scale) {
        Tensor q = q0, k = k0, v = v0, out, lse;
        const Shape s{false, causal, (int)q.size(0), (int)q.size(1), (int)k.size(1), (int)q.size(2), (int)k.size(2), (int)q.size(3), scale};
        if (!forward_rounded(q, k, v, s, out, lse)) {
            std::tie(q, k, v) = std::tuple_cat(bf16(q0, k0, v0));
            std::tie(out, lse) = forward_lse(rows16(q), rows16(k), rows16(v), nullptr, nullptr, s);
        }
        ctx->save_for_backward({q, k, v, out, lse});
        ctx->saved_data["f32"] = (int64_t)f32_bits(q0, k0, v0);
        ctx->saved_data["causal"] = causal;
        ctx->saved_data["scale"] = scale;
        return out;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list dout) {
        const auto t = ctx->get_saved_variables();
        const Tensor &q = t[0], &k = t[1];
        const Shape s{false, ctx->saved_data["causal"].toBool(), (int)q.size(0), (int)q.size(1), (int)k.size(1), (int)q.size(2), (int)k.size(2),
                      (int)q.size(3), ctx->saved_data["scale"].toDouble()};
        auto g = backward_of(q, k, t[2], t[3], dout[0], t[4], nullptr, nullptr, s, (int)ctx->saved_data["f32"].toInt());
        g.resize(5);
        return g;
    }
};
struct PackedFn : torch::autograd::Function<PackedFn> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& cu_q, const Tensor& cu_k,
                          int64_t max_q, int64_t max_k, bool causal, double scale) {
        const auto [q, k, v] = bf16(q0, k0, v0);
        const Shape s{true, causal, (int)cu_q.numel() - 1, (int)q.size(1), (int)k.size(1), (int)max_q, (int)max_k, (int)q.size(2), scale};
        auto [out, lse] = forward_lse(rows16(q), rows16(k), rows16(v), (const int32_t*)cu_q.data_ptr(), (const int32_t*)cu_k.data_ptr(), s);
        ctx->save_for_backward({q, k, v, out, lse, cu_q, cu_k});
        ctx->saved_data["f32"] = (int64_t)f32_bits(q0, k0, v0);
        ctx->saved_data["max_q"] = max_q;
        ctx->saved_data["max_k"] = max_k;
        ctx->saved_data["causal"] = causal;
        ctx->saved_data["scale"] = scale;
        return out;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list dout) {
        const auto t = ctx->get_saved_variables();
        const Tensor &q = t[0], &k = t[1];
        const Shape s{true, ctx->saved_data["causal"].toBool(), (int)t[5].numel() - 1, (int)q.size(1), (int)k.size(1), (int)ctx->saved_data["max_q"].toInt(),
                      (int)ctx->saved_data["max_k"].toInt(), (int)q.size(2), ctx->saved_data["scale"].toDouble()};
        auto g = backward_of(q, k, t[2], t[3], dout[0], t[4], (const int32_t*)t[5].data_ptr(), (const int32_t*)t[6].data_ptr(), s,
                             (int)ctx->saved_data["f32"].toInt());
        g.resize(9);
        return g;
    }
};

// q, k and v of a prefill: bf16 or fp32, not all fp32 (their result depends on autocast), nothing that is broadcast and rounded
bool qkv(Args& a, int64_t dim, const Tensor*& q, const Tensor*& k, const Tensor*& v, bool& grad) {
    const Tensor* t[3] = {a.any(0), a.any(1), a.any(2)};
    int wide = 0;
    grad = false;
    for (const Tensor* x : t) {
        if (!a.ok) return false;
        a.need(x->dim() == dim && x->numel() > 0 && (x->scalar_type() == kBF16 || x->scalar_type() == kF32));
        if (!a.ok) return false;
        if (x->scalar_type() == kF32) {
            ++wide;
            for (int64_t st : x->strides()) a.need(st != 0);
        }
        if (x->requires_grad()) grad = true;
        a.need(!x->_fw_grad(0).defined());
    }
    a.need(wide < 3);
    grad = grad && at::GradMode::is_enabled();
    q = t[0];
    k = t[1];
    v = t[2];
    return a.ok;
}

Tensor forward_only(const Tensor& q, const Tensor& k, const Tensor& v, const int32_t* cu_q, const int32_t* cu_k, const Shape& s, int window, int keep_first) {
    const auto dev = q.device();
    const int64_t rows = s.packed ? q.size(0) : (int64_t)s.B * s.Sq;
    const Tensor out = s.packed ? make(q.sizes(), kBF16, dev) : make({s.B, s.Sq, s.Hq, s.D}, kBF16, dev).permute({0, 2, 1, 3});
    if (window > 0) {
        check(mi355_prefill_fwd_window(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), Strides(q), Strides(k), Strides(v), Strides(out), cu_q, cu_k,
                                       nullptr, nullptr, s.B, s.Hq, s.Hkv, s.Sq, s.Sk, s.D, (float)s.scale, window, keep_first, MI355_BF16, stream_of(dev)),
              "mi355_prefill_fwd_window");
        return out;
    }
    const int splits = mi355_prefill_suggest_prompt_kv_splits(s.B, s.Hq, s.D, s.Sq, s.Sk, rows, s.causal, compute_units(dev));
    if (splits > 1) {
        const Tensor ws = make({std::max<int64_t>((int64_t)mi355_prefill_splitkv_workspace_bytes(rows, s.Hq, s.D, splits), 16)}, at::kByte, dev);
        check(mi355_prefill_fwd_splitkv(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), Strides(q), Strides(k), Strides(v), Strides(out), cu_q, cu_k,
                                        s.B, s.Hq, s.Hkv, s.Sq, s.Sk, s.D, (float)s.scale, s.mode(), MI355_BF16, splits, rows, ws.data_ptr(), bytes(ws),
                                        stream_of(dev)),
              "mi355_prefill_fwd_splitkv");
        return out;
    }
    const int64_t no_mask[3] = {0, 0, 0};
    check(mi355_prefill_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), Strides(q), Strides(k), Strides(v), Strides(out), cu_q, cu_k, nullptr,
                            no_mask, s.B, s.Hq, s.Hkv, s.Sq, s.Sk, s.D, (float)s.scale, s.mode(), MI355_BF16, stream_of(dev)),
          "mi355_prefill_fwd");
    return out;
}

// Few heads of more keys than a wavefront or two have at once run on the kernel that deals keys to wavefronts, behind a launch that rounds.  us with fp32 Q and K, rounded
// on their way in / like this: heads of 64, one of 128 keys 6.0 / 6.4, of 150 7.9 / 6.9, of 256 10.1 / 7.3, 32 of 128 6.2 / 7.2, of 150 8.2 / 7.9, of 256 10.5 / 8.4, 64 of 256 10.6 / 11.1; of 32,
// one of 150 6.0 / 6.2, of 177 6.4 / 6.2, of 256 7.3 / 6.4, 32 of 177 6.8 / 6.8, of 256 7.8 / 7.0, 64 of 256 7.8 / 8.3.  (Causal; without a mask every wavefront has all keys.)
bool keys_dealt(const Shape& s, const c10::Device& dev) {
    return (int64_t)s.B * s.Hq <= (s.causal ? 32 : 64) && s.Sk > (s.D == 64 ? 128 : 176) &&
           mi355_prefill_kernel(s.B, s.Hq, s.Hkv, s.D, s.Sq, s.Sk, s.mode(), 0, 0, 0, 1, 0, compute_units(dev), nullptr) == MI355_PREFILL_KEYS;
}

// forward_only of short heads with fp32 among q, k and v, which the kernel rounds on their way in; undefined: no such form of this call, or not the faster one
Tensor forward_mixed(const Tensor& q, const Tensor& k, const Tensor& v, const Shape& s) {
    const int f32 = f32_bits(q, k, v);
    if (f32 == 0 || !((float)s.scale > 0.f) || !mi355_prefill_fwd_rounds(s.Hq, s.Hkv, s.Sq, s.Sk, s.D, s.mode()) || keys_dealt(s, q.device())) return {};
    for (const Tensor* t : {&q, &k, &v})
        if (!whole_rows(*t) || t->stride(2) <= 0 || t->stride(2) >= (1 << 24)) return {};
    const auto dev = q.device();
    const Tensor out = make({s.B, s.Sq, s.Hq, s.D}, kBF16, dev).permute({0, 2, 1, 3});
    check(mi355_prefill_fwd_rounded(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), Strides(q), Strides(k), Strides(v), Strides(out), f32, s.B, s.Hq,
                                    s.Hkv, s.Sq, s.Sk, s.D, (float)s.scale, s.mode(), stream_of(dev)),
          "mi355_prefill_fwd_rounded");
    return out;
}

// (q, k, v, causal, softmax_scale)
PyObject* prefill(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 5);
    const Tensor *q, *k, *v;
    bool grad;
    if (!a.ok || !qkv(a, 4, q, k, v, grad)) Py_RETURN_NONE;
    const bool causal = a.flag(3);
    a.need(k->size(0) == q->size(0) && k->size(3) == q->size(3) && v->sizes() == k->sizes() && q->size(1) % k->size(1) == 0);
    const double scale = a.none(4) ? 1.0 / std::sqrt((double)q->size(3)) : a.number(4);
    if (!a.plain()) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        if (grad) {
            out = DenseFn::apply(*q, *k, *v, causal, scale);
        } else {
            const Shape s{false, causal, (int)q->size(0), (int)q->size(1), (int)k->size(1), (int)q->size(2), (int)k->size(2), (int)q->size(3), scale};
            out = forward_mixed(*q, *k, *v, s);
            if (!out.defined()) {
                const auto [q16, k16, v16] = bf16(*q, *k, *v);
                out = forward_only(rows16(q16), rows16(k16), rows16(v16), nullptr, nullptr, s, 0, 0);
            }
        }
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

const Tensor* lengths(Args& a, int i) {
    const Tensor* t = a.tensor(i, kI32, 1);
    if (t) a.need(t->is_contiguous());
    return t;
}

// (q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, causal, softmax_scale, window, keep_first)
PyObject* prefill_packed(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 11);
    const Tensor *q, *k, *v;
    bool grad;
    if (!a.ok || !qkv(a, 3, q, k, v, grad)) Py_RETURN_NONE;
    const Tensor *cu_q = lengths(a, 3), *cu_k = lengths(a, 4);
    const int64_t max_q = a.integer(5), max_k = a.integer(6), window = a.integer(9), keep_first = a.integer(10);
    const bool causal = a.flag(7);
    if (!a.ok) Py_RETURN_NONE;
    a.need(cu_q->numel() == cu_k->numel() && cu_q->numel() >= 2 && max_q >= 1 && max_k >= 1 && window >= 0 && keep_first >= 0);
    a.need(k->size(2) == q->size(2) && v->sizes() == k->sizes() && q->size(1) % k->size(1) == 0 && (window == 0 || (causal && !grad)));
    const double scale = a.none(8) ? 1.0 / std::sqrt((double)q->size(2)) : a.number(8);
    if (!a.plain()) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        if (grad) {
            out = PackedFn::apply(*q, *k, *v, *cu_q, *cu_k, max_q, max_k, causal, scale);
        } else {
            const Shape s{true, causal, (int)cu_q->numel() - 1, (int)q->size(1), (int)k->size(1), (int)max_q, (int)max_k, (int)q->size(2), scale};
            const auto [q16, k16, v16] = bf16(*q, *k, *v);
            out = forward_only(rows16(q16), rows16(k16), rows16(v16), (const int32_t*)cu_q->data_ptr(), (const int32_t*)cu_k->data_ptr(), s,
                               (int)window, (int)keep_first);
        }
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- the paged cache --------------------------------------------------------------------------------
struct Cache {
    const Tensor *k, *v, *k_scale = nullptr, *v_scale = nullptr;
    int64_t blocks = 0, heads = 0, D = 0;
    bool fp8() const { return k_scale != nullptr; }
};
bool is_byte(const Tensor& t) { return t.scalar_type() == at::kByte || t.scalar_type() == at::kFloat8_e4m3fn; }
// caches at i and i + 1, their scales (or None twice) at s and s + 1
bool cache(Args& a, int i, int s, Cache& c) {
    c.k = a.any(i);
    c.v = a.any(i + 1);
    if (!a.ok) return false;
    const bool fp8 = s >= 0 && !(a.none(s) && a.none(s + 1));
    for (const Tensor* t : {c.k, c.v}) a.need(t->dim() == 4 && t->size(2) == 16 && t->is_contiguous() && (fp8 ? is_byte(*t) : t->scalar_type() == kBF16));
    a.need(a.ok && c.k->sizes() == c.v->sizes() && c.k->size(1) > 0);
    if (!a.ok) return false;
    c.blocks = c.k->size(0);
    c.heads = c.k->size(1);
    c.D = c.k->size(3);
    if (fp8) {
        c.k_scale = a.whole(s, kF32, {c.blocks, c.heads});
        c.v_scale = a.whole(s + 1, kF32, {c.blocks, c.heads});
    }
    return a.ok;
}
bool tables_of(Args& a, int i, int64_t B, const Tensor*& tables, const Tensor*& lens) {
    tables = a.tensor(i, kI32, 2);
    lens = a.whole(i + 1, kI32, {B});
    if (a.ok) a.need(tables->size(0) == B && tables->stride(1) == 1 && tables->size(1) > 0);
    return a.ok;
}

// (q, k_cache, v_cache, block_tables, context_lens, softmax_scale, k_scale, v_scale, max_context, workspace, window, keep_first)
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 12);
    const Tensor *q = a.tensor(0, kBF16, 3), *tables, *lens, *ws = nullptr;
    Cache c;
    if (!a.ok || !cache(a, 1, 6, c) || !tables_of(a, 3, q->size(0), tables, lens)) Py_RETURN_NONE;
    const int64_t B = q->size(0), H = q->size(1), D = q->size(2), width = tables->size(1) * 16;
    const int64_t longest = a.none(8) ? width : a.integer(8), window = a.integer(10), keep_first = a.integer(11);
    const double scale = a.none(5) ? 1.0 / std::sqrt((double)D) : a.number(5);
    if (!a.none(9)) ws = a.any(9);
    a.need(B > 0 && c.D == D && q->is_contiguous() && Args::aligned(*q) && longest <= width && window >= 0 && keep_first >= 0);
    if (!a.plain()) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        out = make({B, H, D}, kBF16, a.device);
        Tensor own;
        if (!ws) {
            own = make({std::max<int64_t>((int64_t)mi355_paged_decode_workspace_bytes((int)B, (int)H, (int)D, (int)longest), 16)}, at::kByte, a.device);
            ws = &own;
        }
        const int kind = c.fp8() ? MI355_FP8_E4M3 : MI355_BF16;
        if (window > 0)
            check(mi355_paged_decode_fwd_window(q->data_ptr(), H * D, c.k->data_ptr(), c.v->data_ptr(), out.data_ptr(), H * D, (const int32_t*)tables->data_ptr(),
                                                tables->stride(0), (const int32_t*)lens->data_ptr(), (const float*)ptr(c.k_scale), (const float*)ptr(c.v_scale),
                                                nullptr, nullptr, ws->data_ptr(), bytes(*ws), (int)B, (int)H, (int)c.heads, (int)D, 16, c.blocks, (int)longest,
                                                (float)scale, (int)window, (int)keep_first, kind, stream_of(a.device)),
                  "mi355_paged_decode_fwd_window");
        else
            check(mi355_paged_decode_fwd(q->data_ptr(), c.k->data_ptr(), c.v->data_ptr(), out.data_ptr(), (const int32_t*)tables->data_ptr(), tables->stride(0),
                                         (const int32_t*)lens->data_ptr(), (const float*)ptr(c.k_scale), (const float*)ptr(c.v_scale), ws->data_ptr(), bytes(*ws),
                                         (int)B, (int)H, (int)c.heads, (int)D, 16, c.blocks, (int)longest, (float)scale, kind, stream_of(a.device)),
                  "mi355_paged_decode_fwd");
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// (q, k, v, positions, freq_cache, k_cache, v_cache, k_scale, v_scale, slot_mapping, k_out): the rotated q, or (q, k)
PyObject* rope_and_cache(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 11);
    const Tensor *q = a.ok ? a.heads(0, kBF16) : nullptr, *k = a.ok ? a.heads(1, kBF16) : nullptr, *v = a.ok ? a.heads(2, kBF16) : nullptr;
    Cache c;
    if (!a.ok || !cache(a, 5, 7, c)) Py_RETURN_NONE;
    const int64_t T = q->size(0), H = q->size(1), D = q->size(2);
    const Tensor *pos = a.whole(3, kI32, {T}), *freq = a.tensor(4, kF32, 3), *slots = a.whole(9, kI64, {T});
    if (!a.ok) Py_RETURN_NONE;
    const bool k_out = a.flag(10);
    a.need(T > 0 && k->sizes() == v->sizes() && k->size(0) == T && k->size(2) == D && k->size(1) == c.heads && c.D == D);
    a.need(D == 32 || D == 64 || D == 128);
    a.need(freq->size(0) == 2 && freq->size(2) * 2 == D && freq->is_contiguous());
    if (!a.plain()) Py_RETURN_NONE;
    Tensor q_rot, k_rot;
    {
        NoGil released;
        q_rot = make({T, H, D}, kBF16, a.device);
        if (k_out) k_rot = make({T, c.heads, D}, kBF16, a.device);
        void* kr = k_out ? k_rot.data_ptr() : nullptr;
        const int64_t ks = k_out ? k_rot.stride(0) : 0;
        if (c.fp8())
            check(mi355_rope_and_cache_fp8(q->data_ptr(), k->data_ptr(), v->data_ptr(), q_rot.data_ptr(), c.k->data_ptr(), c.v->data_ptr(),
                                           (float*)c.k_scale->data_ptr(), (float*)c.v_scale->data_ptr(), (const float*)freq->data_ptr(),
                                           (const int32_t*)pos->data_ptr(), (const int64_t*)slots->data_ptr(), c.blocks, (int)T, (int)H, (int)c.heads, (int)D,
                                           (int)freq->size(1), q->stride(0), k->stride(0), v->stride(0), q_rot.stride(0), kr, ks, stream_of(a.device)),
                  "mi355_rope_and_cache_fp8");
        else
            check(mi355_rope_and_cache(q->data_ptr(), k->data_ptr(), v->data_ptr(), q_rot.data_ptr(), c.k->data_ptr(), c.v->data_ptr(),
                                       (const float*)freq->data_ptr(), (const int32_t*)pos->data_ptr(), (const int64_t*)slots->data_ptr(), c.blocks, (int)T,
                                       (int)H, (int)c.heads, (int)D, (int)freq->size(1), q->stride(0), k->stride(0), v->stride(0), q_rot.stride(0), kr, ks,
                                       stream_of(a.device)),
                  "mi355_rope_and_cache");
    }
    PyObject* first = THPVariable_Wrap(std::move(q_rot));
    if (!k_out || !first) return first;
    PyObject* second = THPVariable_Wrap(std::move(k_rot));
    PyObject* both = second ? PyTuple_Pack(2, first, second) : nullptr;
    Py_DECREF(first);
    Py_XDECREF(second);
    return both;
    END_HANDLE_TH_ERRORS
}

// (q, k_cache, v_cache, cu_seqlens_q, block_tables, context_lens, max_seqlen_q, softmax_scale, max_context, k_scale, v_scale, total_context,
//  cu_seqlens_k)
PyObject* paged_prefill(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 13);
    const Tensor *q = a.ok ? a.heads(0, kBF16) : nullptr, *tables, *lens, *cu_k = nullptr;
    Cache c;
    if (!a.ok || !cache(a, 1, 9, c)) Py_RETURN_NONE;
    const Tensor* cu_q = lengths(a, 3);
    if (!a.ok || !tables_of(a, 4, cu_q->numel() - 1, tables, lens)) Py_RETURN_NONE;
    const int64_t T = q->size(0), H = q->size(1), D = q->size(2), B = cu_q->numel() - 1, width = tables->size(1) * 16;
    const int64_t max_q = a.integer(6);
    int64_t longest = a.none(8) ? width : a.integer(8);
    const double scale = a.none(7) ? 1.0 / std::sqrt((double)D) : a.number(7);
    a.need(T > 0 && B > 0 && max_q >= 1 && longest >= 1 && c.D == D && (D == 32 || D == 64 || D == 128) && H % c.heads == 0);
    int64_t rows = 0;
    if (a.ok && c.fp8()) {
        longest = std::min(longest, width);
        rows = std::min(a.none(11) ? 0 : a.integer(11), B * longest);
        if (a.none(12)) Py_RETURN_NONE;
        cu_k = a.whole(12, kI32, {B + 1});
        a.need(rows > 0);
    }
    if (!a.plain() || (at::GradMode::is_enabled() && q->requires_grad())) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        if (c.fp8()) {
            const Tensor k = make({rows, c.heads, D}, kBF16, a.device), v = make({rows, c.heads, D}, kBF16, a.device);
            check(mi355_gather_kv_fp8(c.k->data_ptr(), c.v->data_ptr(), (const float*)c.k_scale->data_ptr(), (const float*)c.v_scale->data_ptr(),
                                      (const int32_t*)tables->data_ptr(), tables->stride(0), (longest + 15) / 16, (const int32_t*)lens->data_ptr(),
                                      (const int32_t*)cu_k->data_ptr(), k.data_ptr(), v.data_ptr(), c.heads * D, rows, (int)B, (int)c.heads, (int)D, 16,
                                      c.blocks, stream_of(a.device)),
                  "mi355_gather_kv_fp8");
            const Shape s{true, true, (int)B, (int)H, (int)c.heads, (int)max_q, (int)longest, (int)D, scale};
            out = forward_only(*q, k, v, (const int32_t*)cu_q->data_ptr(), (const int32_t*)cu_k->data_ptr(), s, 0, 0);
        } else {
            out = make({T, H, D}, kBF16, a.device);
            const int splits = mi355_prefill_suggest_kv_splits((int)B, (int)H, (int)D, (int)max_q, (int)longest, T, 1, compute_units(a.device));
            Tensor ws;
            if (splits > 1) ws = make({std::max<int64_t>((int64_t)mi355_prefill_splitkv_workspace_bytes(T, (int)H, (int)D, splits), 16)}, at::kByte, a.device);
            check(mi355_prefill_paged_fwd_headwise(q->data_ptr(), c.k->data_ptr(), c.v->data_ptr(), out.data_ptr(), q->stride(0), out.stride(0),
                                                   (const int32_t*)cu_q->data_ptr(), (const int32_t*)tables->data_ptr(), tables->stride(0), tables->size(1),
                                                   (const int32_t*)lens->data_ptr(), nullptr, nullptr, (int)B, (int)H, (int)c.heads, (int)max_q, (int)D, 16,
                                                   c.blocks, (float)scale, MI355_BF16, splits, T, splits > 1 ? ws.data_ptr() : nullptr,
                                                   splits > 1 ? bytes(ws) : 0, stream_of(a.device)),
                  "mi355_prefill_paged_fwd_headwise");
        }
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- layer operators ----------------------------------------------------------------------------------
int64_t row_stride(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }

// (h, w, bias, top): (ids, weights)
PyObject* moe_route(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 4);
    const Tensor *h = a.ok ? a.matrix(0, kBF16) : nullptr, *w = a.ok ? a.matrix(1, kBF16) : nullptr;
    if (!a.ok) Py_RETURN_NONE;
    const Tensor* bias = a.whole(2, kF32, {w->size(0)});
    const int64_t T = h->size(0), k = h->size(1), top = a.integer(3);
    a.need(T > 0 && w->size(1) == k && top > 0 && top <= w->size(0));
    if (!a.plain()) Py_RETURN_NONE;
    Tensor ids, weights;
    {
        NoGil released;
        ids = make({T, top}, kI32, a.device);
        weights = make({T, top}, kF32, a.device);
        check(mi355_moe_route(h->data_ptr(), w->data_ptr(), (const float*)bias->data_ptr(), (int32_t*)ids.data_ptr(), (float*)weights.data_ptr(), nullptr, T,
                              row_stride(*h), row_stride(*w), (int)k, (int)w->size(0), (int)top, MI355_BF16, stream_of(a.device)),
              "mi355_moe_route");
    }
    PyObject *first = THPVariable_Wrap(std::move(ids)), *second = first ? THPVariable_Wrap(std::move(weights)) : nullptr;
    PyObject* both = second ? PyTuple_Pack(2, first, second) : nullptr;
    Py_XDECREF(first);
    Py_XDECREF(second);
    return both;
    END_HANDLE_TH_ERRORS
}

// (h, ids, weights, w_gate_up, w_down, pairs up to which there is no order)
PyObject* moe_experts(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 6);
    const Tensor *h = a.ok ? a.matrix(0, kBF16) : nullptr, *ids = a.ok ? a.tensor(1, kI32, 2) : nullptr, *down = a.ok ? a.tensor(4, kBF16, 3) : nullptr;
    if (!a.ok) Py_RETURN_NONE;
    const int64_t T = h->size(0), k = h->size(1), top = ids->size(1), E = down->size(0), cols = down->size(1), ff = down->size(2), direct = a.integer(5);
    const Tensor *weights = a.whole(2, kF32, {T, top}), *up = a.whole(3, kBF16, {E, 2 * ff, k});
    a.need(T > 0 && top > 0 && ids->size(0) == T && ids->is_contiguous() && down->is_contiguous());
    if (!a.plain()) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        const int64_t pairs = T * top, padded = (cols + 7) / 8 * 8;                  // (16-byte aligned rows)
        out = make({pairs, padded}, kBF16, a.device);
        if (padded != cols) out = out.narrow(1, 0, cols);
        const Tensor act = make({pairs, ff}, kBF16, a.device);
        void* s = stream_of(a.device);
        if (pairs <= direct) {
            check(mi355_moe_direct(h->data_ptr(), up->data_ptr(), down->data_ptr(), (const int32_t*)ids->data_ptr(), (const float*)weights->data_ptr(),
                                   act.data_ptr(), out.data_ptr(), T, row_stride(*h), out.stride(0), (int)E, (int)top, (int)k, (int)ff, (int)cols, s),
                  "mi355_moe_direct");
        } else {
            const Tensor offsets = make({E + 1}, kI32, a.device), order = make({pairs}, kI32, a.device);
            int32_t *off = (int32_t*)offsets.data_ptr(), *ord = (int32_t*)order.data_ptr();
            check(mi355_moe_group((const int32_t*)ids->data_ptr(), pairs, (int)E, off, ord, s), "mi355_moe_group");
            check(mi355_moe_gate_up(h->data_ptr(), up->data_ptr(), act.data_ptr(), off, ord, T, row_stride(*h), ff, (int)E, (int)top, (int)k, (int)ff, MI355_BF16,
                                    MI355_TILING_AUTO, s),
                  "mi355_moe_gate_up");
            check(mi355_moe_down(act.data_ptr(), down->data_ptr(), (const float*)weights->data_ptr(), out.data_ptr(), off, ord, T, ff, out.stride(0), (int)E,
                                 (int)top, (int)ff, (int)cols, MI355_BF16, MI355_TILING_AUTO, s),
                  "mi355_moe_down");
        }
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// (resid, weight, sub, routed, top, weight_offset, eps) with bf16 sub, routed and result: (x, y)
PyObject* residual_rms(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 7);
    if (!a.ok || a.none(2)) Py_RETURN_NONE;
    const Tensor *sub = a.matrix(2, kBF16), *routed = a.none(3) ? nullptr : a.matrix(3, kBF16);
    if (!a.ok) Py_RETURN_NONE;
    const int64_t T = sub->size(0), d = sub->size(1), top = a.integer(4);
    const Tensor *resid = a.none(0) ? nullptr : a.whole(0, kF32, {T, d}), *weight = a.whole(1, kF32, {d});
    const double offset = a.number(5), eps = a.number(6);
    if (a.ok && routed) a.need(routed->size(0) == T * top && routed->size(1) == d);
    a.need(T > 0 && d > 0);
    if (!a.plain()) Py_RETURN_NONE;
    Tensor x, y;
    {
        NoGil released;
        x = resid ? *resid : make({T, d}, kF32, a.device);
        y = make({T, d}, kBF16, a.device);
        check(mi355_residual_rms_fwd((const float*)ptr(resid), (float*)x.data_ptr(), sub->data_ptr(), ptr(routed), (int)top, nullptr, nullptr, 0,
                                     (const float*)weight->data_ptr(), (float)offset, (float)eps, y.data_ptr(), T, (int)d, (int)d, sub->stride(0),
                                     routed ? routed->stride(0) : 0, d, MI355_BF16, stream_of(a.device)),
              "mi355_residual_rms_fwd");
    }
    PyObject *first = THPVariable_Wrap(std::move(x)), *second = first ? THPVariable_Wrap(std::move(y)) : nullptr;
    PyObject* both = second ? PyTuple_Pack(2, first, second) : nullptr;
    Py_XDECREF(first);
    Py_XDECREF(second);
    return both;
    END_HANDLE_TH_ERRORS
}

// (y, z, weight, groups, eps, out)
PyObject* gated_norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 6);
    const Tensor *y = a.ok ? a.matrix(0, kBF16) : nullptr, *z = a.ok ? a.matrix(1, kBF16) : nullptr;
    if (!a.ok) Py_RETURN_NONE;
    const int64_t T = y->size(0), d = y->size(1), groups = a.integer(3);
    const Tensor *weight = a.whole(2, kF32, {d}), *into = a.none(5) ? nullptr : a.matrix(5, kBF16);
    const double eps = a.number(4);
    if (a.ok && into) a.need(into->sizes() == y->sizes());
    a.need(T > 0 && z->sizes() == y->sizes() && groups >= 1 && d % groups == 0);
    if (!a.plain()) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        out = into ? *into : make({T, d}, kBF16, a.device);
        check(mi355_gated_norm_fwd(y->data_ptr(), z->data_ptr(), (const float*)weight->data_ptr(), out.data_ptr(), T, (int)d, (int)groups, y->stride(0),
                                   z->stride(0), out.stride(0), (float)eps, MI355_BF16, stream_of(a.device)),
              "mi355_gated_norm_fwd");
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// (proj, conv, conv_b, dt_bias, neg_a, d_skip, conv_state, ssm_state, slots, positions, cu_seqlens, xbc_col, dt_col, heads, vdim, state, groups,
//  tokens per segment, tokens of a whole sequence): bf16 prompts, scan chosen by the library
PyObject* ssm_prefill(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 19);
    const Tensor *proj = a.ok ? a.matrix(0, kBF16) : nullptr, *conv = a.ok ? a.tensor(1, kF32, 2) : nullptr, *ring = a.ok ? a.tensor(6, kBF16, 3) : nullptr;
    const Tensor* slots = a.ok ? a.tensor(8, kI32, 1) : nullptr;
    if (!a.ok) Py_RETURN_NONE;
    int64_t v[8];
    for (int i = 0; i < 8; ++i) v[i] = a.integer(11 + i);
    const auto [xbc_col, dt_col, heads, vdim, state, groups, seg_len, whole_len] = v;
    a.need(heads > 0 && vdim > 0 && state > 0 && groups > 0 && seg_len >= 0);
    if (!a.ok) Py_RETURN_NONE;
    const int64_t T = proj->size(0), inner = heads * vdim, channels = inner + 2 * groups * state, taps = conv->size(0), B = slots->size(0);
    const int64_t padded = (vdim + 3) / 4 * 4, n_slots = ring->size(0), width = proj->size(1);
    const Tensor *conv_b = a.whole(2, kF32, {channels}), *dt_bias = a.whole(3, kF32, {heads}), *neg_a = a.whole(4, kF32, {heads}),
                 *d_skip = a.whole(5, kF32, {heads}), *states = a.whole(7, kF32, {n_slots, heads, state, padded}), *pos = a.whole(9, kI32, {T}),
                 *cu = a.whole(10, kI32, {B + 1});
    a.need(T > 0 && B > 0 && conv->size(1) == channels && conv->is_contiguous() && ring->is_contiguous() && ring->size(1) == taps && ring->size(2) == channels &&
           slots->is_contiguous() && xbc_col >= 0 && xbc_col <= width - channels && dt_col >= 0 && dt_col <= width - heads);
    if (!a.plain()) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        out = make({T, inner}, kBF16, a.device);
        const Tensor xbc = make({T, channels}, kBF16, a.device);
        Tensor seg_state, seg_decay;
        if (seg_len > 0) {
            const int64_t units = T / seg_len + B;
            seg_state = make({units, heads, state, vdim}, kF32, a.device);
            seg_decay = make({units, heads}, kF32, a.device);
        }
        mi355_ssm_args s{};
        s.proj = proj->data_ptr();
        s.conv_weight = (const float*)conv->data_ptr();
        s.conv_bias = (const float*)conv_b->data_ptr();
        s.dt_bias = (const float*)dt_bias->data_ptr();
        s.neg_a = (const float*)neg_a->data_ptr();
        s.d_skip = (const float*)d_skip->data_ptr();
        s.conv_state = ring->data_ptr();
        s.ssm_state = (float*)states->data_ptr();
        s.slots = (const int32_t*)slots->data_ptr();
        s.positions = (const int32_t*)pos->data_ptr();
        s.cu_seqlens = (const int32_t*)cu->data_ptr();
        s.xbc = xbc.data_ptr();
        s.y = out.data_ptr();
        s.proj_row_stride = row_stride(*proj);
        s.xbc_col = xbc_col;
        s.dt_col = dt_col;
        s.y_row_stride = inner;
        s.n_rows = T;
        s.batch = (int)B;
        s.heads = (int)heads;
        s.vdim = (int)vdim;
        s.state = (int)state;
        s.groups = (int)groups;
        s.taps = (int)taps;
        s.n_slots = (int)n_slots;
        s.dtype = MI355_BF16;
        s.seg_state = seg_len > 0 ? (float*)seg_state.data_ptr() : nullptr;
        s.seg_decay = seg_len > 0 ? (float*)seg_decay.data_ptr() : nullptr;
        s.seg_len = (int)seg_len;
        s.whole_len = (int)whole_len;
        check(mi355_ssm_prefill(&s, MI355_SCAN_AUTO, stream_of(a.device)), "mi355_ssm_prefill");
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// x or rows of it, and its residual: what rows_linear and rows_qkv share
struct Rows {
    const Tensor *x, *w, *norm, *ids;
    int64_t T = 0, k = 0;
};
bool rows_of(Args& a, int x, int w, int norm, int ids, Rows& r) {
    r.x = a.ok ? a.tensor(x, kBF16, 2) : nullptr;
    r.w = a.ok ? a.tensor(w, kBF16, 2) : nullptr;
    if (!a.ok) return false;
    r.k = r.w->size(1);
    r.ids = a.none(ids) ? nullptr : a.tensor(ids, kI64, 1);
    r.norm = a.none(norm) ? nullptr : a.whole(norm, kF32, {r.k});
    if (!a.ok) return false;
    r.T = r.ids ? r.ids->size(0) : r.x->size(0);
    a.need(r.T > 0 && r.x->size(0) > 0 && r.x->size(1) == r.k && r.x->stride(1) == 1 && r.w->is_contiguous() && (!r.ids || r.ids->is_contiguous()));
    return a.ok;
}
mi355_rows_args rows_args(const Rows& r, const Tensor& out, int64_t out_stride, int64_t n, double eps) {
    mi355_rows_args s{};
    s.x = r.x->data_ptr();
    s.x_rows = (const int64_t*)ptr(r.ids);
    s.norm = (const float*)ptr(r.norm);
    s.w = r.w->data_ptr();
    s.out = out.data_ptr();
    s.x_count = r.x->size(0);
    s.x_row_stride = row_stride(*r.x);
    s.out_row_stride = out_stride;
    s.eps = (float)eps;
    s.n_rows = (int)r.T;
    s.n = (int)n;
    s.k = (int)r.k;
    return s;
}

// (x, w, norm, eps, x_rows, resid, resid_rows, gate_up, fp32 result, prompt)
PyObject* rows_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 10);
    Rows r;
    if (!rows_of(a, 0, 1, 2, 4, r)) Py_RETURN_NONE;
    const double eps = a.number(3);
    const Tensor *resid = a.none(5) ? nullptr : a.tensor(5, kBF16, 2), *resid_ids = a.none(6) ? nullptr : a.whole(6, kI64, {r.T});
    const bool gate_up = a.flag(7), f32 = a.flag(8), prompt = a.flag(9);
    if (!a.ok) Py_RETURN_NONE;
    const int64_t cols = r.w->size(0) / (gate_up ? 2 : 1);
    a.need((resid != nullptr) + gate_up + f32 <= 1 && (resid || !resid_ids) && (!gate_up || r.w->size(0) % 2 == 0) && cols > 0);
    if (resid) a.need(resid->size(1) == cols && resid->stride(1) == 1 && (resid_ids || resid->size(0) == r.T) && resid->size(0) > 0);
    if (!a.plain()) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        out = make({r.T, cols}, f32 ? kF32 : kBF16, a.device);
        mi355_rows_args s = rows_args(r, out, cols, cols, eps);
        if (resid) {
            s.resid = resid->data_ptr();
            s.resid_rows = (const int64_t*)ptr(resid_ids);
            s.resid_count = resid->size(0);
            s.resid_row_stride = row_stride(*resid);
        }
        const int mode = resid ? MI355_ROWS_ADD : gate_up ? MI355_ROWS_GATE_UP : f32 ? MI355_ROWS_F32 : MI355_ROWS_STORE;
        if (prompt) check(mi355_prompt_linear(&s, mode, stream_of(a.device)), "mi355_prompt_linear");
        else check(mi355_rows_linear(&s, mode, stream_of(a.device)), "mi355_rows_linear");
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// (x, w, positions, freq_cache, k_cache, v_cache, slot_mapping, n_q_heads, norm, eps, x_rows)
PyObject* rows_qkv(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Args a(args, n, 11);
    Rows r;
    Cache c;
    if (!rows_of(a, 0, 1, 8, 10, r) || !cache(a, 4, -1, c)) Py_RETURN_NONE;
    const Tensor *pos = a.whole(2, kI32, {r.T}), *freq = a.tensor(3, kF32, 3), *slots = a.whole(6, kI64, {r.T});
    const int64_t heads = a.integer(7);
    const double eps = a.number(9);
    if (!a.ok) Py_RETURN_NONE;
    a.need(heads > 0 && r.w->size(0) == (heads + 2 * c.heads) * c.D && freq->size(0) == 2 && freq->size(2) * 2 == c.D && freq->is_contiguous());
    if (!a.plain()) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil released;
        out = make({r.T, heads, c.D}, kBF16, a.device);
        mi355_rows_args s = rows_args(r, out, heads * c.D, r.w->size(0), eps);
        s.k_cache = c.k->data_ptr();
        s.v_cache = c.v->data_ptr();
        s.slots = (const int64_t*)slots->data_ptr();
        s.positions = (const int32_t*)pos->data_ptr();
        s.freq_cache = (const float*)freq->data_ptr();
        s.num_blocks = c.blocks;
        s.n_q_heads = (int)heads;
        s.n_kv_heads = (int)c.heads;
        s.head_dim = (int)c.D;
        s.context_length = (int)freq->size(1);
        check(mi355_rows_linear(&s, MI355_ROWS_QKV, stream_of(a.device)), "mi355_rows_linear");
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

#define CALL(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CALL(prefill),     CALL(prefill_packed), CALL(decode),       CALL(rope_and_cache), CALL(paged_prefill), CALL(moe_route),
                         CALL(moe_experts), CALL(residual_rms),   CALL(gated_norm),   CALL(ssm_prefill),    CALL(rows_linear), CALL(rows_qkv),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&module); }
