// q4_binding.cpp -- the Python mirror's hot calls in native code.
//
// At one token the kernels take 3-10 us, and the ctypes route in __init__.py
// takes 12-15 us of host time per call: a tensor check is several Python
// attribute reads (five to eight tensors a call), each weight a ctypes
// structure, the current stream and the new output a torch call each.  Here
// the same checks run on the C++ tensors.  Each function takes its Python
// counterpart's arguments by position and returns its result, or None for
// anything that is not the plain accepted call (other types, sizes the checks
// reject, tensor subclasses, active torch function or dispatch modes): the
// caller then runs its own checks, which raise the errors or make the call.
// Nothing is kept between calls but the library's entry points.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include "swiftltx_q4.h"

namespace {

// The library's entry points, by the address ctypes loaded them at.
#define SLTX_ENTRIES(X)                                                                           \
    X(sltx_matmul_q4) X(sltx_matmul_q4_fast) X(sltx_matmul_q4_fast_f32) X(sltx_silu_mul)          \
    X(sltx_linear) X(sltx_matmul_q4_silu_mul) X(sltx_matmul_q4_ex) X(sltx_matmul_q4_geglu)        \
    X(sltx_embedding_q4) X(sltx_rms_norm) X(sltx_residual_rms_norm) X(sltx_rmsnorm_matmul_q4)     \
    X(sltx_residual_rmsnorm_matmul_q4_silu_mul) X(sltx_matmul_q4_residual)                        \
    X(sltx_matmul_q4_residual_rms_norm) X(sltx_argmax) X(sltx_sample_top_p)
#define X(name) decltype(&name) f_##name = nullptr;
SLTX_ENTRIES(X)
#undef X

PyObject* g_check = nullptr;        // __init__.check: raises for a status
PyTypeObject* g_weight = nullptr;   // Q4Weight
PyObject *s_weight, *s_scales, *s_biases, *s_K, *s_group_size, *s_cuda_stream;

// Not the plain accepted call: the Python code takes it from here.
struct Decline {};

void need(bool ok) {
    if (!ok) throw Decline{};
}

const at::Tensor& tensor(PyObject* o) {
    need(THPVariable_CheckExact(o));
    return THPVariable_Unpack(o);
}

int32_t i32(PyObject* o) {
    need(PyLong_CheckExact(o));
    int over = 0;
    const long v = PyLong_AsLongAndOverflow(o, &over);
    need(!over && v >= INT32_MIN && v <= INT32_MAX);
    return (int32_t)v;
}

float f32(PyObject* o) {
    need(PyFloat_CheckExact(o));
    return (float)PyFloat_AS_DOUBLE(o);
}

// A device tensor of dtype d, contiguous, of at least count elements: its
// address (as _need checks it).
void* data(const at::Tensor& t, at::ScalarType d, int64_t count) {
    need(t.is_cuda() && t.scalar_type() == d && t.is_contiguous() && t.numel() >= count);
    return t.data_ptr();
}
void* data(PyObject* o, at::ScalarType d, int64_t count) { return data(tensor(o), d, count); }

bool shape_ok(int32_t K, int32_t g) {
    return K > 0 && K % 32 == 0 && (g == 32 || g == 64 || g == 128) && K % g == 0;
}

const uint32_t* words(PyObject* o, int64_t count) {
    const at::Tensor& t = tensor(o);
    need(t.scalar_type() == at::kInt || t.scalar_type() == at::kUInt32);
    return static_cast<const uint32_t*>(data(t, t.scalar_type(), count));
}

int32_t attr_i32(PyObject* o, PyObject* name) {
    PyObject* a = PyObject_GetAttr(o, name);
    if (!a) {
        PyErr_Clear();
        throw Decline{};
    }
    struct Drop { PyObject* p; ~Drop() { Py_DECREF(p); } } d{a};
    return i32(a);
}

// A Q4Weight of N rows.  Its tensors stay referenced by it for the call.
sltx_q4_weight weight(PyObject* o, int32_t N) {
    need(Py_TYPE(o) == g_weight && N > 0);
    sltx_q4_weight w{};
    w.K = attr_i32(o, s_K);
    w.group_size = attr_i32(o, s_group_size);
    need(shape_ok(w.K, w.group_size));
    const int64_t groups = (int64_t)N * (w.K / w.group_size);
    PyObject* a[3] = {PyObject_GetAttr(o, s_weight), PyObject_GetAttr(o, s_scales),
                      PyObject_GetAttr(o, s_biases)};
    struct Drop { PyObject** a; ~Drop() { for (int i = 0; i < 3; ++i) Py_XDECREF(a[i]); } } d{a};
    if (!a[0] || !a[1] || !a[2]) {
        PyErr_Clear();
        throw Decline{};
    }
    w.weight = words(a[0], (int64_t)N * w.K / 8);
    w.scales = static_cast<const uint16_t*>(data(a[1], at::kHalf, groups));
    w.biases = static_cast<const uint16_t*>(data(a[2], at::kHalf, groups));
    return w;
}

int32_t dtype_code(at::ScalarType d) {
    need(d == at::kHalf || d == at::kBFloat16 || d == at::kFloat);
    return d == at::kHalf ? SLTX_F16 : d == at::kBFloat16 ? SLTX_BF16 : SLTX_F32;
}

// Without the interpreter lock while it lives.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    Unlocked() = default;
    Unlocked(const Unlocked&) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// The output the caller gave, or a new one: the object to return (owned) and
// the address.  torch's allocator may wait for the GPU (to give cached blocks
// back before it asks for more), so it runs without the interpreter lock, as
// torch.empty runs it.
struct Out {
    PyObject* obj = nullptr;
    void* ptr = nullptr;
    Out() = default;
    Out(const Out&) = delete;
    ~Out() { Py_XDECREF(obj); }
    PyObject* give() {
        PyObject* o = obj;
        obj = nullptr;
        return o;
    }
    void set(PyObject* o, at::IntArrayRef shape, at::ScalarType d, const at::Tensor& like) {
        int64_t n = 1;
        for (int64_t s : shape) n *= s;
        if (o == Py_None) {
            need(like.is_cuda());
            at::Tensor t;
            {
                Unlocked unlocked;
                t = at::empty(shape, at::TensorOptions().dtype(d).device(like.device()));
            }
            ptr = t.data_ptr();
            obj = THPVariable_Wrap(std::move(t));
            if (!obj) throw Decline{};
        } else {
            ptr = data(o, d, n);
            Py_INCREF(o);
            obj = o;
        }
    }
};

void* stream(PyObject* o) {
    if (o == Py_None) return c10::hip::getCurrentHIPStream().stream();
    if (PyLong_CheckExact(o)) {
        void* st = PyLong_AsVoidPtr(o);
        need(!PyErr_Occurred());
        return st;
    }
    PyObject* a = PyObject_GetAttr(o, s_cuda_stream);
    if (!a) {
        PyErr_Clear();
        throw Decline{};
    }
    const bool ok = PyLong_CheckExact(a);
    void* st = ok ? PyLong_AsVoidPtr(a) : nullptr;
    Py_DECREF(a);
    need(ok && !PyErr_Occurred());
    return st;
}

// The library call without the interpreter lock (as ctypes makes it); false
// with the Python error set where it failed.
template <typename F>
bool call(F&& f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    if (rc == SLTX_OK) return true;
    PyObject* r = PyObject_CallFunction(g_check, "i", rc);
    Py_XDECREF(r);
    if (r) PyErr_Format(PyExc_RuntimeError, "status %d", rc);
    return false;
}

PyObject* pair_of(Out& a, Out& b) {
    PyObject* t = PyTuple_Pack(2, a.obj, b.obj);
    return t;
}

// body with the number of arguments it expects; None where it declines.
template <typename F>
PyObject* guarded(Py_ssize_t n, Py_ssize_t want, F&& body) {
    try {
        need(g_check && n == want && !at::impl::torch_function_mode_enabled() &&
             !c10::impl::TorchDispatchModeTLS::any_modes_set());
        return body();
    } catch (...) {
        // declined, or a torch error (say, a tensor without storage): the
        // Python code meets it again
        if (PyErr_Occurred()) PyErr_Clear();
        Py_RETURN_NONE;
    }
}

#define ENTRY(name) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)

// x, weight, scales, biases, M, K, N, group_size, out, stream
template <typename F>
PyObject* matmul(F f, at::ScalarType d, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 10, [&]() -> PyObject* {
        const int32_t M = i32(a[4]), K = i32(a[5]), N = i32(a[6]), g = i32(a[7]);
        need(M > 0 && N > 0 && shape_ok(K, g));
        const void* x = data(a[0], at::kHalf, (int64_t)M * K);
        const uint32_t* w = words(a[1], (int64_t)N * K / 8);
        const auto* s = static_cast<const uint16_t*>(data(a[2], at::kHalf, (int64_t)N * (K / g)));
        const auto* b = static_cast<const uint16_t*>(data(a[3], at::kHalf, (int64_t)N * (K / g)));
        Out out;
        out.set(a[8], {M, N}, d, tensor(a[0]));
        void* st = stream(a[9]);
        return call([&] { return f(x, w, s, b, out.ptr, M, K, N, g, st); }) ? out.give() : nullptr;
    });
}

ENTRY(py_matmul_q4) { return matmul(f_sltx_matmul_q4, at::kHalf, a, n); }
ENTRY(py_matmul_q4_fast) { return matmul(f_sltx_matmul_q4_fast, at::kHalf, a, n); }
ENTRY(py_matmul_q4_fast_f32) {
    return matmul([](const void* x, const uint32_t* w, const uint16_t* s, const uint16_t* b, void* o, int32_t M,
                     int32_t K, int32_t N, int32_t g, void* st) {
        return f_sltx_matmul_q4_fast_f32(x, w, s, b, static_cast<float*>(o), M, K, N, g, st);
    }, at::kFloat, a, n);
}

// a, b, out, stream
ENTRY(py_silu_mul) {
    return guarded(n, 4, [&]() -> PyObject* {
        const at::Tensor& t = tensor(a[0]);
        const int64_t count = t.numel();
        need(count > 0);
        const void *x = data(t, at::kHalf, count), *y = data(a[1], at::kHalf, count);
        Out out;
        out.set(a[2], t.sizes(), at::kHalf, t);
        void* st = stream(a[3]);
        return call([&] { return f_sltx_silu_mul(x, y, out.ptr, count, st); }) ? out.give() : nullptr;
    });
}

// x, w, M, K, N, fast, out, stream
ENTRY(py_linear) {
    return guarded(n, 8, [&]() -> PyObject* {
        const int32_t M = i32(a[2]), K = i32(a[3]), N = i32(a[4]);
        need(M > 0 && (a[5] == Py_True || a[5] == Py_False));
        const sltx_q4_weight w = weight(a[1], N);
        need(w.K == K);
        const void* x = data(a[0], at::kHalf, (int64_t)M * K);
        Out out;
        out.set(a[6], {M, N}, at::kHalf, tensor(a[0]));
        void* st = stream(a[7]);
        const int fast = a[5] == Py_True;
        return call([&] { return f_sltx_linear(x, &w, out.ptr, M, K, N, fast, st); }) ? out.give() : nullptr;
    });
}

// x, gate, up, M, K, N, out, stream
template <typename F>
PyObject* gated(F f, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 8, [&]() -> PyObject* {
        const int32_t M = i32(a[3]), K = i32(a[4]), N = i32(a[5]);
        need(M > 0);
        const sltx_q4_weight g = weight(a[1], N), u = weight(a[2], N);
        need(g.K == K && u.K == K);
        const void* x = data(a[0], at::kHalf, (int64_t)M * K);
        Out out;
        out.set(a[6], {M, N}, at::kHalf, tensor(a[0]));
        void* st = stream(a[7]);
        return call([&] { return f(x, &g, &u, out.ptr, M, K, N, st); }) ? out.give() : nullptr;
    });
}
ENTRY(py_matmul_q4_silu_mul) { return gated(f_sltx_matmul_q4_silu_mul, a, n); }
ENTRY(py_matmul_q4_geglu) { return gated(f_sltx_matmul_q4_geglu, a, n); }

// x, w, M, N, out_dtype, bias, epilogue, out, stream
ENTRY(py_matmul_q4_ex) {
    return guarded(n, 9, [&]() -> PyObject* {
        const int32_t M = i32(a[2]), N = i32(a[3]), epilogue = i32(a[6]);
        need(M > 0 && (a[4] == Py_None || THPDtype_Check(a[4])));
        const at::ScalarType want = a[4] == Py_None ? at::kFloat : reinterpret_cast<THPDtype*>(a[4])->scalar_type;
        const sltx_q4_weight w = weight(a[1], N);
        const at::Tensor& xt = tensor(a[0]);
        const int32_t xd = dtype_code(xt.scalar_type());
        const void* x = data(xt, xt.scalar_type(), (int64_t)M * w.K);
        const auto* bias = a[5] == Py_None ? nullptr : static_cast<const float*>(data(a[5], at::kFloat, N));
        const at::ScalarType od = a[7] == Py_None ? want : tensor(a[7]).scalar_type();
        const int32_t oc = dtype_code(od);
        Out out;
        out.set(a[7], {M, N}, od, xt);
        void* st = stream(a[8]);
        return call([&] { return f_sltx_matmul_q4_ex(x, xd, &w, bias, epilogue, out.ptr, oc, M, N, st); })
                   ? out.give() : nullptr;
    });
}

// x, weight, eps, rows, dim, out, stream
ENTRY(py_rms_norm) {
    return guarded(n, 7, [&]() -> PyObject* {
        const float eps = f32(a[2]);
        const int32_t rows = i32(a[3]), dim = i32(a[4]);
        need(rows > 0 && dim > 0);
        const void* x = data(a[0], at::kHalf, (int64_t)rows * dim);
        const auto* w = static_cast<const float*>(data(a[1], at::kFloat, dim));
        Out out;
        out.set(a[5], {rows, dim}, at::kHalf, tensor(a[0]));
        void* st = stream(a[6]);
        return call([&] { return f_sltx_rms_norm(x, w, eps, out.ptr, rows, dim, st); }) ? out.give() : nullptr;
    });
}

// a, b, weight, eps, rows, dim, residual_out, norm_out, stream
ENTRY(py_residual_rms_norm) {
    return guarded(n, 9, [&]() -> PyObject* {
        const float eps = f32(a[3]);
        const int32_t rows = i32(a[4]), dim = i32(a[5]);
        need(rows > 0 && dim > 0);
        const int64_t count = (int64_t)rows * dim;
        const void *x = data(a[0], at::kHalf, count), *y = data(a[1], at::kHalf, count);
        const auto* w = static_cast<const float*>(data(a[2], at::kFloat, dim));
        Out res, norm;
        res.set(a[6], {rows, dim}, at::kHalf, tensor(a[0]));
        norm.set(a[7], {rows, dim}, at::kHalf, tensor(a[0]));
        void* st = stream(a[8]);
        return call([&] { return f_sltx_residual_rms_norm(x, y, w, eps, res.ptr, norm.ptr, rows, dim, st); })
                   ? pair_of(res, norm) : nullptr;
    });
}

// x, norm_weight, eps, w, N, out, stream
ENTRY(py_rmsnorm_matmul_q4) {
    return guarded(n, 7, [&]() -> PyObject* {
        const float eps = f32(a[2]);
        const int32_t N = i32(a[4]);
        const sltx_q4_weight w = weight(a[3], N);
        const void* x = data(a[0], at::kHalf, w.K);
        const auto* nw = static_cast<const float*>(data(a[1], at::kFloat, w.K));
        Out out;
        out.set(a[5], {1, N}, at::kHalf, tensor(a[0]));
        void* st = stream(a[6]);
        return call([&] { return f_sltx_rmsnorm_matmul_q4(x, nw, eps, &w, out.ptr, N, st); }) ? out.give() : nullptr;
    });
}

// a, b, norm_weight, eps, gate, up, N, residual_out, out, stream
ENTRY(py_residual_rmsnorm_matmul_q4_silu_mul) {
    return guarded(n, 10, [&]() -> PyObject* {
        const float eps = f32(a[3]);
        const int32_t N = i32(a[6]);
        const sltx_q4_weight g = weight(a[4], N), u = weight(a[5], N);
        const void *x = data(a[0], at::kHalf, g.K), *y = data(a[1], at::kHalf, g.K);
        const auto* nw = static_cast<const float*>(data(a[2], at::kFloat, g.K));
        Out res, out;
        res.set(a[7], {1, g.K}, at::kHalf, tensor(a[0]));
        out.set(a[8], {1, N}, at::kHalf, tensor(a[0]));
        void* st = stream(a[9]);
        return call([&] {
                   return f_sltx_residual_rmsnorm_matmul_q4_silu_mul(x, y, nw, eps, res.ptr, &g, &u, out.ptr, N, st);
               }) ? pair_of(res, out) : nullptr;
    });
}

// x, w, residual, M, N, out, stream
ENTRY(py_matmul_q4_residual) {
    return guarded(n, 7, [&]() -> PyObject* {
        const int32_t M = i32(a[3]), N = i32(a[4]);
        need(M > 0);
        const sltx_q4_weight w = weight(a[1], N);
        const void *x = data(a[0], at::kHalf, (int64_t)M * w.K), *r = data(a[2], at::kHalf, (int64_t)M * N);
        Out out;
        out.set(a[5], {M, N}, at::kHalf, tensor(a[0]));
        void* st = stream(a[6]);
        return call([&] { return f_sltx_matmul_q4_residual(x, &w, r, out.ptr, M, N, st); }) ? out.give() : nullptr;
    });
}

// x, w, residual, norm_weight, eps, M, N, sum_rounded, residual_out, norm_out, stream
ENTRY(py_matmul_q4_residual_rms_norm) {
    return guarded(n, 11, [&]() -> PyObject* {
        const float eps = f32(a[4]);
        const int32_t M = i32(a[5]), N = i32(a[6]);
        need(M > 0 && (a[7] == Py_True || a[7] == Py_False));
        const sltx_q4_weight w = weight(a[1], N);
        const void *x = data(a[0], at::kHalf, (int64_t)M * w.K), *r = data(a[2], at::kHalf, (int64_t)M * N);
        const auto* nw = static_cast<const float*>(data(a[3], at::kFloat, N));
        Out res, norm;
        res.set(a[8], {M, N}, at::kHalf, tensor(a[0]));
        norm.set(a[9], {M, N}, at::kHalf, tensor(a[0]));
        void* st = stream(a[10]);
        const int rounded = a[7] == Py_True;
        return call([&] {
                   return f_sltx_matmul_q4_residual_rms_norm(x, &w, r, nw, eps, M, N, rounded, res.ptr, norm.ptr, st);
               }) ? pair_of(res, norm) : nullptr;
    });
}

// table, vocab, token_ids, out, stream
ENTRY(py_embedding_q4) {
    return guarded(n, 5, [&]() -> PyObject* {
        const int32_t vocab = i32(a[1]);
        const sltx_q4_weight t = weight(a[0], vocab);
        const at::Tensor& ids = tensor(a[2]);
        need(ids.numel() > 0 && ids.numel() <= INT32_MAX);
        const int32_t count = (int32_t)ids.numel();
        const auto* id = static_cast<const int32_t*>(data(ids, at::kInt, count));
        Out out;
        out.set(a[3], {count, t.K}, at::kHalf, ids);
        void* st = stream(a[4]);
        return call([&] { return f_sltx_embedding_q4(&t, vocab, id, count, out.ptr, st); }) ? out.give() : nullptr;
    });
}

// fp16 / fp32 logits: address, dtype code and count
const void* logits_of(PyObject* o, int32_t* code, int32_t* count) {
    const at::Tensor& t = tensor(o);
    need((t.scalar_type() == at::kHalf || t.scalar_type() == at::kFloat) && t.numel() <= INT32_MAX);
    *code = dtype_code(t.scalar_type());
    *count = (int32_t)t.numel();
    return data(t, t.scalar_type(), *count);
}

// logits, out, stream
ENTRY(py_argmax) {
    return guarded(n, 3, [&]() -> PyObject* {
        int32_t code, count;
        const void* l = logits_of(a[0], &code, &count);
        Out out;
        out.set(a[1], {1}, at::kInt, tensor(a[0]));
        void* st = stream(a[2]);
        return call([&] { return f_sltx_argmax(l, code, count, static_cast<int32_t*>(out.ptr), st); })
                   ? out.give() : nullptr;
    });
}

// logits, temperature, top_p, repetition_penalty, seen_tokens, u, out, stream
ENTRY(py_sample) {
    return guarded(n, 8, [&]() -> PyObject* {
        int32_t code, count, n_seen = 0;
        const void* l = logits_of(a[0], &code, &count);
        const float t = f32(a[1]), p = f32(a[2]), pen = f32(a[3]), u = f32(a[5]);
        const int32_t* seen = nullptr;
        if (a[4] != Py_None) {
            const at::Tensor& s = tensor(a[4]);
            need(s.numel() > 0 && s.numel() <= INT32_MAX);
            n_seen = (int32_t)s.numel();
            seen = static_cast<const int32_t*>(data(s, at::kInt, n_seen));
        }
        Out out;
        out.set(a[6], {1}, at::kInt, tensor(a[0]));
        void* st = stream(a[7]);
        return call([&] {
                   return f_sltx_sample_top_p(l, code, count, t, p, pen, seen, n_seen, u,
                                              static_cast<int32_t*>(out.ptr), st);
               }) ? out.give() : nullptr;
    });
}

// init(addresses by name, check, Q4Weight)
PyObject* py_init(PyObject*, PyObject* args) {
    PyObject *addr, *check, *type;
    if (!PyArg_ParseTuple(args, "O!OO!", &PyDict_Type, &addr, &check, &PyType_Type, &type)) return nullptr;
#define X(name)                                                                              \
    {                                                                                        \
        PyObject* v = PyDict_GetItemString(addr, #name);                                     \
        if (!v) return PyErr_Format(PyExc_KeyError, "no address of %s", #name);              \
        f_##name = reinterpret_cast<decltype(&::name)>(PyLong_AsVoidPtr(v));                 \
        if (PyErr_Occurred()) return nullptr;                                                \
    }
    SLTX_ENTRIES(X)
#undef X
    Py_INCREF(check);
    Py_INCREF(type);
    Py_XSETREF(g_check, check);
    PyObject* old = reinterpret_cast<PyObject*>(g_weight);
    g_weight = reinterpret_cast<PyTypeObject*>(type);
    Py_XDECREF(old);
    Py_RETURN_NONE;
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"init", py_init, METH_VARARGS, nullptr},
    METHOD(matmul_q4), METHOD(matmul_q4_fast), METHOD(matmul_q4_fast_f32), METHOD(silu_mul),
    METHOD(linear), METHOD(matmul_q4_silu_mul), METHOD(matmul_q4_geglu), METHOD(matmul_q4_ex),
    METHOD(rms_norm), METHOD(residual_rms_norm), METHOD(rmsnorm_matmul_q4),
    METHOD(residual_rmsnorm_matmul_q4_silu_mul), METHOD(matmul_q4_residual),
    METHOD(matmul_q4_residual_rms_norm), METHOD(embedding_q4), METHOD(argmax), METHOD(sample),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_q4_binding", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__q4_binding(void) {
    s_weight = PyUnicode_InternFromString("weight");
    s_scales = PyUnicode_InternFromString("scales");
    s_biases = PyUnicode_InternFromString("biases");
    s_K = PyUnicode_InternFromString("K");
    s_group_size = PyUnicode_InternFromString("group_size");
    s_cuda_stream = PyUnicode_InternFromString("cuda_stream");
    return PyModule_Create(&module);
}
