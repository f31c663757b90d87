// h3mi._fast: the common calls of the h3mi Python functions, from tensors to the
// C ABI without Python in between.
//
// A call from Python through ctypes costs 10-14 us of host time (tensor checks,
// allocation, the stream lookup, argument conversion), 27 for the two launches
// of a W8A8 linear: more than the kernels of a short call.  Here the same checks,
// allocations and launches take 4-9 us.
//
// Every function returns None without doing anything unless its arguments are
// what the Python function accepts in its plain form: exact torch tensors on one
// GPU, with the types, shapes and strides checked here, none of them wrapped by a
// transform, and no torch-function mode active.  The Python function then runs
// its own checks, so every other form, and every error, is decided there.  A
// dispatch mode sees the allocations of either path, and nothing else of them.
// A nonzero status of the C ABI raises the H3miError that the Python path raises.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <stdlib.h>
#include <string.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/h3mi.h"

namespace {

PyObject* g_error = nullptr;  // h3mi._lib.H3miError
int64_t g_shape[3] = {0, 0, 0};
bool g_shape_set = false;     // (M, N, K) of the last GEMM through here, for best_config

// Keys of tensors whose memory is not simply theirs to read (subclasses and
// modes, functorch wrappers, functionalization, lazy conjugation and negation).
const c10::DispatchKeySet kWrapped({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                    c10::DispatchKey::PythonDispatcher, c10::DispatchKey::Functionalize,
                                    c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                    c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::Batched,
                                    c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                    c10::DispatchKey::ZeroTensor});

// The tensors of one call: each must be a plain strided GPU tensor on the
// first one's device.
struct Args {
    c10::Device dev{c10::kCPU};
    bool ok = !at::impl::torch_function_mode_enabled();

    const at::Tensor* any(PyObject* o) {
        if (!ok) return nullptr;
        ok = false;
        if (!THPVariable_CheckExact(o)) return nullptr;
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(kWrapped)) return nullptr;
        if (dev.is_cpu()) dev = t.device();
        if (t.device() != dev || t.numel() == 0) return nullptr;
        ok = true;
        return &t;
    }
    const at::Tensor* typed(PyObject* o, c10::ScalarType type) {
        const at::Tensor* t = any(o);
        if (t && t->scalar_type() != type) ok = false;
        return t;
    }
    // contiguous, with n elements
    const at::Tensor* flat(PyObject* o, c10::ScalarType type, int64_t n) {
        const at::Tensor* t = typed(o, type);
        if (t && (t->numel() != n || !t->is_contiguous())) ok = false;
        return t;
    }
    // contiguous [rows, n]; rows < 0: any number, returned
    const at::Tensor* table(PyObject* o, int64_t n, int64_t* rows) {
        const at::Tensor* t = typed(o, c10::kBFloat16);
        if (!t) return nullptr;
        if (!t->is_contiguous() || t->numel() % n != 0 || (*rows >= 0 && t->numel() / n != *rows)) ok = false;
        *rows = t->numel() / n;
        return t;
    }
    // 2-D with unit column stride
    const at::Tensor* rows2(PyObject* o, c10::ScalarType type, bool contiguous) {
        const at::Tensor* t = typed(o, type);
        if (t && (t->dim() != 2 || t->stride(1) != 1 || (contiguous && !t->is_contiguous()))) ok = false;
        return t;
    }
    at::Tensor empty(at::IntArrayRef size, c10::ScalarType type) const {
        return at::empty(size, at::TensorOptions().dtype(type).device(dev));
    }
    void* stream() const { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }
};

const uint16_t* u16(const at::Tensor* t) { return t ? static_cast<const uint16_t*>(t->data_ptr()) : nullptr; }
uint16_t* mu16(const at::Tensor& t) { return static_cast<uint16_t*>(t.data_ptr()); }
const float* f32(const at::Tensor* t) { return static_cast<const float*>(t->data_ptr()); }

PyObject* raise_status(int status) {
    const char* msg = h3mi_last_error();
    PyObject* e = PyObject_CallFunction(g_error, "is", status, msg ? msg : "");
    if (e) {
        PyErr_SetObject(g_error, e);
        Py_DECREF(e);
    }
    return nullptr;
}

// A float or int; anything else is the Python function's to convert.
bool number(PyObject* o, double* v) {
    if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
    *v = PyFloat_AsDouble(o);
    if (*v != -1.0 || !PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

PyObject* pair(const at::Tensor& a, const at::Tensor& b) {
    PyObject *x = THPVariable_Wrap(a), *y = x ? THPVariable_Wrap(b) : nullptr;
    PyObject* r = y ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    return r;
}

// H3_LINEAR_FAST_ALLCFG=1 tunes every shape: the Python function's work.
bool tuning() {
    const char* v = getenv("H3_LINEAR_FAST_ALLCFG");
    return v && strcmp(v, "1") == 0;
}

// A GEMM's operands beside xq and xs.
struct Gemm {
    const at::Tensor *w, *ws, *bias = nullptr;
    int64_t N = 0;
    Gemm(Args& a, PyObject* wo, PyObject* wso, PyObject* bo, int64_t K) {
        w = a.rows2(wo, c10::kChar, true);
        if (!a.ok) return;
        N = w->size(0);
        if (w->size(1) != K) a.ok = false;
        ws = a.flat(wso, c10::kFloat, N);
        if (bo != Py_None) bias = a.flat(bo, c10::kBFloat16, N);
    }
    int run(const int8_t* xq, const float* xs, const at::Tensor& out, int64_t M, int64_t K, int64_t ldx, void* st) const {
        return h3mi_w8a8_gemm_bf16(xq, static_cast<const int8_t*>(w->data_ptr()), xs, f32(ws), u16(bias), mu16(out), M, N, K,
                                   ldx, w->stride(0), out.stride(0), st);
    }
};

void note_shape(int64_t M, int64_t N, int64_t K) {
    g_shape[0] = M, g_shape[1] = N, g_shape[2] = K;
    g_shape_set = true;
}

#define H3MI_BEGIN HANDLE_TH_ERRORS
#define H3MI_END END_HANDLE_TH_ERRORS
#define H3MI_ARGS(COUNT) \
    if (n != (COUNT)) {  \
        PyErr_SetString(PyExc_TypeError, "h3mi._fast: wrong number of arguments"); \
        return nullptr;  \
    }

// (x, weight, weight_scale, bias)
PyObject* w8a8_linear(PyObject*, PyObject* const* v, Py_ssize_t n) {
    H3MI_BEGIN
    H3MI_ARGS(4)
    Args a;
    const at::Tensor* x = a.rows2(v[0], c10::kBFloat16, false);
    if (!a.ok || tuning()) Py_RETURN_NONE;
    const int64_t M = x->size(0), K = x->size(1);
    const Gemm g(a, v[1], v[2], v[3], K);
    if (!a.ok) Py_RETURN_NONE;
    note_shape(M, g.N, K);
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        const at::Tensor q = a.empty({M, K}, c10::kChar), s = a.empty({M, 1}, c10::kFloat);
        int8_t* const xq = static_cast<int8_t*>(q.data_ptr());
        float* const xs = static_cast<float*>(s.data_ptr());
        out = a.empty({M, g.N}, c10::kBFloat16);
        void* const st = a.stream();
        rc = h3mi_quant_rowwise_i8(u16(x), xq, xs, M, K, x->stride(0), st);
        if (!rc) rc = g.run(xq, xs, out, M, K, K, st);
    }
    return rc ? raise_status(rc) : THPVariable_Wrap(out);
    H3MI_END
}

// (xq, w, xs, ws, bias)
PyObject* int8_mm_scaled(PyObject*, PyObject* const* v, Py_ssize_t n) {
    H3MI_BEGIN
    H3MI_ARGS(5)
    Args a;
    const at::Tensor* xq = a.rows2(v[0], c10::kChar, true);
    if (!a.ok || tuning()) Py_RETURN_NONE;
    const int64_t M = xq->size(0), K = xq->size(1);
    const at::Tensor* xs = a.flat(v[2], c10::kFloat, M);
    const Gemm g(a, v[1], v[3], v[4], K);
    if (!a.ok) Py_RETURN_NONE;
    note_shape(M, g.N, K);
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        out = a.empty({M, g.N}, c10::kBFloat16);
        rc = g.run(static_cast<const int8_t*>(xq->data_ptr()), f32(xs), out, M, K, xq->stride(0), a.stream());
    }
    return rc ? raise_status(rc) : THPVariable_Wrap(out);
    H3MI_END
}

// (x, act): act < 0 the per-token quantizer, else ConvRot's input activation
PyObject* quantize(PyObject*, PyObject* const* v, Py_ssize_t n) {
    H3MI_BEGIN
    H3MI_ARGS(2)
    Args a;
    const at::Tensor* x = a.rows2(v[0], c10::kBFloat16, false);
    if (!a.ok) Py_RETURN_NONE;
    const long act = PyLong_AsLong(v[1]);
    if (act == -1 && PyErr_Occurred()) return nullptr;
    const int64_t M = x->size(0), kin = x->size(1), K = act == H3MI_ACT_SWIGLU ? kin / 2 : kin;
    if (K == 0 || (act == H3MI_ACT_SWIGLU && kin % 2)) Py_RETURN_NONE;
    at::Tensor q, s;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        q = a.empty({M, K}, c10::kChar);
        s = a.empty({M, 1}, c10::kFloat);
        int8_t* const qp = static_cast<int8_t*>(q.data_ptr());
        float* const sp = static_cast<float*>(s.data_ptr());
        rc = act < 0 ? h3mi_quant_rowwise_i8(u16(x), qp, sp, M, K, x->stride(0), a.stream())
                     : h3mi_quant_convrot_i8(u16(x), qp, sp, M, K, x->stride(0), 256, static_cast<int>(act), a.stream());
    }
    return rc ? raise_status(rc) : pair(q, s);
    H3MI_END
}

// The norms' operands: x [S, N], then (gated) o and g, w, ridx, s1, sh.
struct Norm {
    const at::Tensor *x, *o = nullptr, *g = nullptr, *w = nullptr, *ridx, *s1 = nullptr, *sh = nullptr;
    int64_t S = 0, N = 0, R = -1;
    Norm(Args& a, PyObject* xo) {
        x = a.rows2(xo, c10::kBFloat16, true);
        if (a.ok) S = x->size(0), N = x->size(1);
    }
    void gate(Args& a, PyObject* oo, PyObject* go) {
        if (!a.ok) return;
        o = a.rows2(oo, c10::kBFloat16, true);
        if (a.ok && (o->size(0) != S || o->size(1) != N)) a.ok = false;
        g = a.table(go, N, &R);
    }
    void rows(Args& a, PyObject* ro) { ridx = a.ok ? a.flat(ro, c10::kInt, S) : nullptr; }
    void norm(Args& a, PyObject* wo, PyObject* s1o, PyObject* sho) {
        if (!a.ok) return;
        w = a.flat(wo, c10::kBFloat16, N);
        s1 = a.table(s1o, N, &R);
        sh = a.table(sho, N, &R);
    }
    const int32_t* ri() const { return static_cast<const int32_t*>(ridx->data_ptr()); }
};

// (x, w, eps, ridx, s1, sh, quant) or (x, o, g, w, eps, ridx, s1, sh, quant)
template <bool GATE>
PyObject* norm_any(PyObject*, PyObject* const* v, Py_ssize_t n) {
    H3MI_BEGIN
    H3MI_ARGS(GATE ? 9 : 7)
    constexpr int B = GATE ? 2 : 0;
    Args a;
    Norm t(a, v[0]);
    if constexpr (GATE) t.gate(a, v[1], v[2]);
    t.rows(a, v[B + 3]);
    t.norm(a, v[B + 1], v[B + 4], v[B + 5]);
    const bool quant = v[B + 6] == Py_True;
    if (!a.ok || (quant && (t.N % 8 || t.N > 8192))) Py_RETURN_NONE;
    double eps;
    if (!number(v[B + 2], &eps)) Py_RETURN_NONE;
    at::Tensor h, qs;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        const float e = static_cast<float>(eps);
        uint16_t* const x = mu16(*t.x);
        if (quant) {
            h = a.empty({t.S, t.N}, c10::kChar);
            qs = a.empty({t.S, 1}, c10::kFloat);
            int8_t* const qp = static_cast<int8_t*>(h.data_ptr());
            float* const sp = static_cast<float*>(qs.data_ptr());
            rc = GATE ? h3mi_gate_norm_mod_quant_i8(x, u16(t.o), u16(t.g), u16(t.w), t.ri(), u16(t.s1), u16(t.sh), nullptr, qp,
                                                    sp, t.S, t.N, t.R, e, a.stream())
                      : h3mi_norm_mod_quant_i8(x, u16(t.w), t.ri(), u16(t.s1), u16(t.sh), nullptr, qp, sp, t.S, t.N, t.R, e,
                                               a.stream());
        } else {
            h = a.empty({t.S, t.N}, c10::kBFloat16);
            rc = GATE ? h3mi_gate_norm_mod_bf16(x, u16(t.o), u16(t.g), u16(t.w), t.ri(), u16(t.s1), u16(t.sh), mu16(h), t.S,
                                                t.N, t.R, e, a.stream())
                      : h3mi_norm_mod_bf16(x, u16(t.w), t.ri(), u16(t.s1), u16(t.sh), mu16(h), t.S, t.N, t.R, e, a.stream());
        }
    }
    if (rc) return raise_status(rc);
    return quant ? pair(h, qs) : THPVariable_Wrap(h);
    H3MI_END
}

// (x, o, g, ridx) -> x
PyObject* gate_(PyObject*, PyObject* const* v, Py_ssize_t n) {
    H3MI_BEGIN
    H3MI_ARGS(4)
    Args a;
    Norm t(a, v[0]);
    t.gate(a, v[1], v[2]);
    t.rows(a, v[3]);
    if (!a.ok) Py_RETURN_NONE;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        rc = h3mi_gate_bf16(mu16(*t.x), u16(t.o), u16(t.g), t.ri(), t.S, t.N, t.R, a.stream());
    }
    if (rc) return raise_status(rc);
    Py_INCREF(v[0]);
    return v[0];
    H3MI_END
}

// q or k as [s, heads, dim] with contiguous heads
struct Heads {
    const at::Tensor* t;
    int64_t S = 0, H = 0, D = 0, ld = 0;
    Heads(Args& a, PyObject* o) {
        t = a.typed(o, c10::kBFloat16);
        if (!a.ok) return;
        const int64_t b = t->dim() == 4 ? 1 : 0;
        if (t->dim() != 3 + b || (b && t->size(0) != 1)) {
            a.ok = false;
            return;
        }
        S = t->size(b), H = t->size(b + 1), D = t->size(b + 2);
        if (t->stride(b + 2) != 1 || (H > 1 && t->stride(b + 1) != D)) a.ok = false;
        ld = S > 1 ? t->stride(b) : H * D;
    }
};

// (q, k, rope_freqs, qw, kw, epsilon, rot_dim) -> (q, k); hardware rsqrt
PyObject* rms_rope_(PyObject*, PyObject* const* v, Py_ssize_t n) {
    H3MI_BEGIN
    H3MI_ARGS(7)
    Args a;
    const Heads q(a, v[0]);
    const Heads k(a, v[1]);
    const at::Tensor* tab = a.typed(v[2], c10::kBFloat16);
    if (!a.ok || k.S != q.S || k.H != q.H || k.D != q.D || !tab->is_contiguous() || tab->dim() < 4) Py_RETURN_NONE;
    const int64_t d = tab->dim(), rot = tab->size(d - 3) * 2;
    if (tab->size(d - 4) != q.S || tab->size(d - 2) != 2 || tab->size(d - 1) != 2 || tab->numel() != q.S * rot * 2)
        Py_RETURN_NONE;
    if (v[6] != Py_None) {
        const long long want = PyLong_AsLongLong(v[6]);
        if (want == -1 && PyErr_Occurred()) PyErr_Clear();
        if (want != rot) Py_RETURN_NONE;
    }
    const at::Tensor *qw = a.flat(v[3], c10::kBFloat16, q.D), *kw = a.flat(v[4], c10::kBFloat16, q.D);
    if (!a.ok) Py_RETURN_NONE;
    double eps;
    if (!number(v[5], &eps)) Py_RETURN_NONE;
    int rc;
    {
        pybind11::gil_scoped_release nogil;
        rc = h3mi_rms_rope_split_half_bf16(mu16(*q.t), mu16(*k.t), u16(tab), u16(qw), u16(kw), q.S, q.H, q.D, q.ld, k.ld, rot,
                                           static_cast<float>(eps), H3MI_RSQRT_HW, nullptr, a.stream());
    }
    return rc ? raise_status(rc) : PyTuple_Pack(2, v[0], v[1]);
    H3MI_END
}

// (set,): set False forgets the last GEMM's shape; returns it, or None
PyObject* last_shape(PyObject*, PyObject* const* v, Py_ssize_t n) {
    H3MI_ARGS(1)
    if (v[0] == Py_False) g_shape_set = false;
    if (!g_shape_set) Py_RETURN_NONE;
    return Py_BuildValue("(LLL)", static_cast<long long>(g_shape[0]), static_cast<long long>(g_shape[1]),
                         static_cast<long long>(g_shape[2]));
}

PyObject* set_error(PyObject*, PyObject* cls) {
    Py_INCREF(cls);
    Py_XDECREF(g_error);
    g_error = cls;
    Py_RETURN_NONE;
}

#define H3MI_FN(NAME, F) {NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(F)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    H3MI_FN("w8a8_linear", &w8a8_linear), H3MI_FN("int8_mm_scaled", &int8_mm_scaled), H3MI_FN("quantize", &quantize),
    H3MI_FN("norm_mod", &norm_any<false>), H3MI_FN("gate_norm_mod_", &norm_any<true>), H3MI_FN("gate_", &gate_),
    H3MI_FN("rms_rope_", &rms_rope_), H3MI_FN("last_shape", &last_shape),
    {"set_error", set_error, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) { return PyModule_Create(&kModule); }
