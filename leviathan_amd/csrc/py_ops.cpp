// The per-call work of leviathan_amd/ops.py in native code: tensor checks, output allocation and the call itself.
//
// A small operator (a 9 MB GEMV is 3.6 us of kernel) is bound by the host that enqueues it.  Of 5.3 us a call the launch
// itself is 2.4; ctypes' conversion of ten arguments and the tensor attributes read from Python were the other half.
// Here the arguments are read through the C API: 3.4 us a call, its kernel the bound again (GEMV 4096 x
// 4096 5.4 -> 3.5 us); a five-operator FFN of 4096/12288 on int8 enqueues in 20 us where it took 35.
//
// Every function takes its arguments by position, None for one that is left out, the context's handle first; the Python
// methods hold names and defaults.  A failed call raises the exception that ops.py registered, built from the status.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>

#include <algorithm>

#include "../../include/leviathan_hip.h"

namespace {

struct Raised {};   // a Python exception is set

PyObject *g_error = nullptr;   // callable(status, message) -> exception

constexpr at::ScalarType kU8 = at::kByte, kI8 = at::kChar, kI32 = at::kInt, kF16 = at::kHalf, kF32 = at::kFloat;

const char *dtype_name(at::ScalarType t) {
    switch (t) {
        case kU8: return "torch.uint8";
        case kI8: return "torch.int8";
        case kI32: return "torch.int32";
        case kF16: return "torch.float16";
        default: return "torch.float32";
    }
}

[[noreturn]] void raise_status(int st, const char *message) {
    PyObject *e = PyObject_CallFunction(g_error, "is", st, message);
    if (e) {
        PyErr_SetObject(reinterpret_cast<PyObject *>(Py_TYPE(e)), e);
        Py_DECREF(e);
    }
    throw Raised{};
}

class Args {
public:
    Args(PyObject *const *v, Py_ssize_t n, Py_ssize_t want) : v_(v) {
        if (n != want) {
            PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
            throw Raised{};
        }
    }
    PyObject *object(int i) const { return v_[i]; }
    bool given(int i) const { return v_[i] != Py_None; }
    bool flag(int i) const {
        const int r = PyObject_IsTrue(v_[i]);
        if (r < 0) throw Raised{};
        return r != 0;
    }
    // A contiguous tensor of that type on the GPU.
    const at::Tensor &tensor(int i, at::ScalarType type, const char *what) const {
        if (THPVariable_Check(v_[i])) {
            const at::Tensor &t = THPVariable_Unpack(v_[i]);
            if (t.is_cuda() && t.scalar_type() == type && t.is_contiguous()) return t;
        }
        PyErr_Format(PyExc_TypeError, "%s: expected a contiguous %s tensor on the GPU", what, dtype_name(type));
        throw Raised{};
    }
    // Any tensor, its type taken on trust (an output buffer, a raw view of weights).
    const at::Tensor &buffer(int i) const {
        if (!THPVariable_Check(v_[i])) {
            PyErr_SetString(PyExc_TypeError, "expected a tensor");
            throw Raised{};
        }
        return THPVariable_Unpack(v_[i]);
    }
    void *optional(int i) const { return given(i) ? buffer(i).data_ptr() : nullptr; }
    float *optional(int i, const char *what) const {
        return given(i) ? static_cast<float *>(tensor(i, kF32, what).data_ptr()) : nullptr;
    }
    uint64_t u64(int i) const {
        const uint64_t r = PyLong_AsUnsignedLongLongMask(v_[i]);
        if (r == (uint64_t)-1 && PyErr_Occurred()) throw Raised{};
        return r;
    }
    uint32_t u32(int i) const { return (uint32_t)u64(i); }
    float f32(int i) const {
        const double r = PyFloat_AsDouble(v_[i]);
        if (r == -1.0 && PyErr_Occurred()) throw Raised{};
        return (float)r;
    }
    lev_ctx *context() const {
        void *p = given(0) ? PyLong_AsVoidPtr(v_[0]) : nullptr;
        if (!p && PyErr_Occurred()) throw Raised{};
        return static_cast<lev_ctx *>(p);
    }

private:
    PyObject *const *v_;
};

// An argument that the caller may leave out, in which case it is allocated.
class Out {
public:
    Out(const Args &a, int i, at::ScalarType type, at::IntArrayRef shape, const at::Tensor &like) {
        if (a.given(i)) {
            object_ = a.object(i);
            t_ = a.buffer(i);
        } else {
            t_ = at::empty(shape, like.options().dtype(type));
        }
    }
    Out(at::ScalarType type, at::IntArrayRef shape, const at::Tensor &like) : t_(at::empty(shape, like.options().dtype(type))) {}
    const at::Tensor &tensor() const { return t_; }
    template <typename T = void>
    T *data() const { return static_cast<T *>(t_.data_ptr()); }
    size_t count() const { return (size_t)t_.numel(); }
    PyObject *result() const {   // a new reference: the caller's own object where it gave one
        if (!object_) return THPVariable_Wrap(t_);
        Py_INCREF(object_);
        return object_;
    }

private:
    PyObject *object_ = nullptr;
    at::Tensor t_;
};

template <typename... O>
PyObject *tuple_of(const O &...outs) {
    PyObject *r = PyTuple_New(sizeof...(outs));
    if (!r) throw Raised{};
    Py_ssize_t i = 0;
    (PyTuple_SET_ITEM(r, i++, outs.result()), ...);
    return r;
}

// Calls without the interpreter's lock, as ctypes does, and raises what it reports.
template <typename F, typename... A>
void call(F fn, lev_ctx *ctx, A... args) {
    int st;
    Py_BEGIN_ALLOW_THREADS
    st = fn(ctx, args...);
    Py_END_ALLOW_THREADS
    if (st != LEV_OK) raise_status(st, lev_hip_last_error(ctx));
}

int64_t at_least_1(uint32_t n) { return std::max<int64_t>(n, 1); }
float *floats(const at::Tensor &t) { return static_cast<float *>(t.data_ptr()); }

// ctx, w, x, in_dim, out_rows, y, w_off, x_count
PyObject *q4_0_gemv(const Args &a) {
    const at::Tensor &w = a.tensor(1, kU8, "w"), &x = a.tensor(2, kF32, "x");
    const uint32_t in_dim = a.u32(3), rows = a.u32(4);
    Out y(a, 5, kF32, {at_least_1(rows)}, w);
    call(lev_hip_q4_0_gemv, a.context(), w.data_ptr(), (size_t)w.numel(), a.u64(6), floats(x),
         a.given(7) ? (size_t)a.u64(7) : (size_t)x.numel(), y.data<float>(), y.count(), in_dim, rows);
    return y.result();
}

// ctx, w, x, in_dim, out_rows, y, w_off, argmax
PyObject *q6_k_gemv(const Args &a) {
    const at::Tensor &w = a.tensor(1, kU8, "w"), &x = a.tensor(2, kF32, "x");
    const uint32_t in_dim = a.u32(3), rows = a.u32(4);
    Out y(a, 5, kF32, {at_least_1(rows)}, w);
    if (!a.flag(7)) {
        call(lev_hip_q6_k_gemv, a.context(), w.data_ptr(), (size_t)w.numel(), a.u64(6), floats(x), (size_t)x.numel(),
             y.data<float>(), y.count(), in_dim, rows, nullptr, nullptr);
        return y.result();
    }
    Out idx(kI32, {1}, w), margin(kF32, {1}, w);
    call(lev_hip_q6_k_gemv, a.context(), w.data_ptr(), (size_t)w.numel(), a.u64(6), floats(x), (size_t)x.numel(),
         y.data<float>(), y.count(), in_dim, rows, idx.data<uint32_t>(), margin.data<float>());
    return tuple_of(y, idx, margin);
}

// ctx, w, x, in_dim, rows, ncol, gain, eps, y, w_off
template <auto FN>
PyObject *gemv_ncol(const Args &a) {
    const at::Tensor &w = a.tensor(1, kU8, "w"), &x = a.tensor(2, kF32, "x");
    const uint32_t in_dim = a.u32(3), rows = a.u32(4), ncol = a.u32(5);
    const float *gain = a.optional(6, "gain");
    Out y(a, 8, kF32, {at_least_1(ncol), at_least_1(rows)}, w);
    call(FN, a.context(), w.data_ptr(), (size_t)w.numel(), a.u64(9), floats(x), (size_t)x.numel(), gain, a.f32(7),
         y.data<float>(), y.count(), in_dim, rows, ncol);
    return y.result();
}

// ctx, x, n, ncol, gain, eps, add, want_y
PyObject *norm_quant_q8(const Args &a) {
    const at::Tensor &x = a.tensor(1, kF32, "x");
    const uint32_t n = a.u32(2), ncol = a.u32(3);
    const float *gain = a.optional(4, "gain"), *add = a.optional(6, "add");
    Out xq(kI8, {at_least_1(ncol), at_least_1(n)}, x), xs(kF32, {at_least_1(ncol), at_least_1(n / 32), 2}, x);
    if (!a.flag(7)) {
        call(lev_hip_norm_quant_q8, a.context(), floats(x), (size_t)x.numel(), add, gain, a.f32(5), xq.data<int8_t>(),
             xs.data<float>(), nullptr, n, ncol);
        return tuple_of(xq, xs);
    }
    Out y(kF32, x.sizes(), x);
    call(lev_hip_norm_quant_q8, a.context(), floats(x), (size_t)x.numel(), add, gain, a.f32(5), xq.data<int8_t>(),
         xs.data<float>(), y.data<float>(), n, ncol);
    return tuple_of(xq, xs, y);
}

// ctx, w, xq, xs, in_dim, rows, ncol, y, w_off
template <auto FN>
PyObject *gemv_q8(const Args &a) {
    const at::Tensor &w = a.tensor(1, kU8, "w"), &xq = a.tensor(2, kI8, "xq"), &xs = a.tensor(3, kF32, "xs");
    const uint32_t in_dim = a.u32(4), rows = a.u32(5), ncol = a.u32(6);
    Out y(a, 7, kF32, {at_least_1(ncol), at_least_1(rows)}, w);
    call(FN, a.context(), w.data_ptr(), (size_t)w.numel(), a.u64(8), static_cast<const int8_t *>(xq.data_ptr()), floats(xs),
         (size_t)xq.numel(), y.data<float>(), y.count(), in_dim, rows, ncol);
    return y.result();
}

// ctx, gate, up, want_act
PyObject *swiglu_quant_q8(const Args &a) {
    const at::Tensor &gate = a.tensor(1, kF32, "gate"), &up = a.tensor(2, kF32, "up");
    const size_t n = (size_t)gate.numel();
    Out xq(kI8, {std::max<int64_t>(n, 1)}, gate), xs(kF32, {std::max<int64_t>(n / 32, 1), 2}, gate);
    if (!a.flag(3)) {
        call(lev_hip_swiglu_quant_q8, a.context(), floats(gate), floats(up), n, xq.data<int8_t>(), xs.data<float>(), nullptr);
        return tuple_of(xq, xs);
    }
    Out act(kF32, gate.sizes(), gate);
    call(lev_hip_swiglu_quant_q8, a.context(), floats(gate), floats(up), n, xq.data<int8_t>(), xs.data<float>(),
         act.data<float>());
    return tuple_of(xq, xs, act);
}

// ctx, w, x_f16, in_dim, rows, tokens, y, w_off
template <auto FN>
PyObject *gemm_prefill(const Args &a) {
    const at::Tensor &w = a.tensor(1, kU8, "w"), &x = a.tensor(2, kF16, "x");
    const uint32_t in_dim = a.u32(3), rows = a.u32(4), tokens = a.u32(5);
    Out y(a, 6, kF32, {at_least_1(tokens), at_least_1(rows)}, w);
    call(FN, a.context(), w.data_ptr(), (size_t)w.numel(), a.u64(7), static_cast<const uint16_t *>(x.data_ptr()),
         (size_t)x.numel(), y.data<float>(), y.count(), in_dim, rows, tokens);
    return y.result();
}

// ctx, x, n, vectors, weight, eps, y
PyObject *rmsnorm(const Args &a) {
    const at::Tensor &x = a.tensor(1, kF32, "x");
    Out y(a, 6, kF32, x.sizes(), x);
    call(lev_hip_rmsnorm, a.context(), floats(x), y.data<float>(), a.u32(2), a.u32(3), static_cast<float *>(a.optional(4)),
         a.f32(5));
    return y.result();
}

// ctx, gu, n, y
PyObject *gelu_up(const Args &a) {
    const at::Tensor &gu = a.tensor(1, kF32, "gu");
    const uint32_t n = a.u32(2);
    Out y(a, 3, kF32, {at_least_1(n)}, gu);
    call(lev_hip_gelu_up, a.context(), floats(gu), y.data<float>(), n);
    return y.result();
}

// ctx, x, y, c, n
PyObject *axpy(const Args &a) {
    const at::Tensor &x = a.tensor(1, kF32, "x"), &y = a.tensor(2, kF32, "y");
    call(lev_hip_axpy, a.context(), floats(x), static_cast<float *>(y.data_ptr()), a.f32(3), a.u32(4));
    Py_INCREF(a.object(2));
    return a.object(2);
}

// ctx, x, ffn_norm, gate_w, up_w, down_w, post_norm, eps, h, gu, act, shared, hidden, inter
PyObject *shared_expert_ffn(const Args &a) {
    const at::Tensor &x = a.tensor(1, kF32, "x"), &h = a.tensor(8, kF32, "h"), &gu = a.tensor(9, kF32, "gu"),
                     &act = a.tensor(10, kF32, "act"), &shared = a.tensor(11, kF32, "shared");
    const at::Tensor &gate = a.tensor(3, kU8, "gate_w"), &up = a.tensor(4, kU8, "up_w"), &down = a.tensor(5, kU8, "down_w");
    const uint32_t hidden = a.u32(12), inter = a.u32(13);
    auto fail = [](int st, const char *fmt, long long p, long long q) {
        char msg[128];
        snprintf(msg, sizeof msg, fmt, p, q);
        raise_status(st, msg);
    };
    if (h.numel() != hidden || act.numel() != inter)
        fail(LEV_ERR_WRONG_INPUT_COUNT, "shared expert: h %lld, act %lld values", h.numel(), act.numel());
    if (gu.numel() < 2 * (int64_t)inter || shared.numel() < hidden)
        fail(LEV_ERR_BAD_DIMENSIONS, "shared expert: gu %lld, shared %lld values", gu.numel(), shared.numel());
    auto out = [](const at::Tensor &t) { return static_cast<float *>(t.data_ptr()); };
    call(lev_hip_shared_expert_ffn_q4_0, a.context(), floats(x), static_cast<float *>(a.optional(2)), gate.data_ptr(),
         (size_t)gate.numel(), up.data_ptr(), (size_t)up.numel(), down.data_ptr(), (size_t)down.numel(),
         static_cast<float *>(a.optional(6)), a.f32(7), out(h), out(gu), out(act), out(shared), hidden, inter);
    Py_RETURN_NONE;
}

// ctx, logits, vocab, ncol
PyObject *argmax(const Args &a) {
    const at::Tensor &logits = a.tensor(1, kF32, "logits");
    const uint32_t vocab = a.u32(2), ncol = a.u32(3);
    Out idx(kI32, {at_least_1(ncol)}, logits), margin(kF32, {at_least_1(ncol)}, logits);
    call(lev_hip_argmax, a.context(), floats(logits), vocab, ncol, idx.data<uint32_t>(), margin.data<float>());
    return tuple_of(idx, margin);
}

// ctx, pools (the struct's bytes), router_w, x, top_k, tokens, expert_scale, y, ids, weights, noalloc
PyObject *moe_layer_q4_0(const Args &a) {
    Py_buffer view;
    if (PyObject_GetBuffer(a.object(1), &view, PyBUF_SIMPLE) != 0) throw Raised{};
    if ((size_t)view.len < sizeof(lev_moe_experts)) {
        PyBuffer_Release(&view);
        PyErr_SetString(PyExc_TypeError, "pools: expected the struct that moe_pools returns");
        throw Raised{};
    }
    lev_moe_experts pools;
    memcpy(&pools, view.buf, sizeof pools);
    PyBuffer_Release(&view);
    const at::Tensor &x = a.tensor(3, kF32, "x");
    const uint32_t top_k = a.u32(4), tokens = a.u32(5);
    const float *router = static_cast<const float *>(a.optional(2)), *scale = static_cast<const float *>(a.optional(6));
    Out y(a, 7, kF32, {at_least_1(tokens), (int64_t)pools.hidden}, x);
    Out ids(a, 8, kI32, {at_least_1(tokens), at_least_1(top_k)}, x), weights(a, 9, kF32, {at_least_1(tokens), at_least_1(top_k)}, x);
    call(a.flag(10) ? lev_hip_moe_layer_q4_0_noalloc : lev_hip_moe_layer_q4_0, a.context(), &pools, router, scale, floats(x),
         y.data<float>(), ids.data<int32_t>(), weights.data<float>(), top_k, tokens);
    return tuple_of(y, ids, weights);
}

// ctx, program handle
PyObject *program_run(const Args &a) {
    void *p = a.given(1) ? PyLong_AsVoidPtr(a.object(1)) : nullptr;
    if (!p && PyErr_Occurred()) throw Raised{};
    call(lev_hip_program_run, a.context(), static_cast<lev_program *>(p));
    Py_RETURN_NONE;
}

template <PyObject *(*F)(const Args &), int N>
PyObject *entry(PyObject *, PyObject *const *v, Py_ssize_t n) {
    try {
        return F(Args(v, n, N));
    } catch (const Raised &) {
    } catch (const std::exception &e) {   // an allocation of torch's
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

PyObject *set_error(PyObject *, PyObject *callable) {
    Py_INCREF(callable);
    Py_XDECREF(g_error);
    g_error = callable;
    Py_RETURN_NONE;
}

template <PyObject *(*F)(const Args &), int N>
constexpr PyMethodDef method(const char *name) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&entry<F, N>)), METH_FASTCALL, nullptr};
}

PyMethodDef g_methods[] = {
    {"set_error", set_error, METH_O, nullptr},
    method<q4_0_gemv, 8>("q4_0_gemv"),
    method<q6_k_gemv, 8>("q6_k_gemv"),
    method<gemv_ncol<lev_hip_q4_k_gemv_ncol>, 10>("q4_k_gemv_ncol"),
    method<gemv_ncol<lev_hip_q6_k_gemv_ncol>, 10>("q6_k_gemv_ncol"),
    method<norm_quant_q8, 8>("norm_quant_q8"),
    method<gemv_q8<lev_hip_q4_k_gemv_q8>, 9>("q4_k_gemv_q8"),
    method<gemv_q8<lev_hip_q6_k_gemv_q8>, 9>("q6_k_gemv_q8"),
    method<swiglu_quant_q8, 4>("swiglu_quant_q8"),
    method<gemm_prefill<lev_hip_q4_k_gemm_prefill>, 8>("q4_k_gemm_prefill"),
    method<gemm_prefill<lev_hip_q6_k_gemm_prefill>, 8>("q6_k_gemm_prefill"),
    method<rmsnorm, 7>("rmsnorm"),
    method<gelu_up, 4>("gelu_up"),
    method<axpy, 5>("axpy"),
    method<shared_expert_ffn, 14>("shared_expert_ffn"),
    method<argmax, 4>("argmax"),
    method<moe_layer_q4_0, 11>("moe_layer_q4_0"),
    method<program_run, 2>("program_run"),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_lev_ops", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__lev_ops(void) { return PyModule_Create(&g_module); }
