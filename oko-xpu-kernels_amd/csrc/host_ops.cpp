// The host path of the Python API's hot calls (xpu_kernels.int8 linear, ffn, the
// backward's products and the quantizer) as a CPython extension: argument
// checks, the packed weight's lookup, allocations and the library call in
// native code.  In Python these cost more than the small calls' kernels: linear
// at 16 x 4096 x 4096 took 17.6 us of host time for 8.5 us of GPU work, 6.9 of
// them the library's two launches.
//
// Every function takes the plain case only -- dense CUDA tensors of exactly the
// dtype, shape, alignment and device the kernels read, no subclass, no
// functorch wrapper, no torch-function or dispatch mode -- and returns None for
// anything else, so that the caller's Python path converts, refuses or computes
// it as before.  Results, and the kernels that run, are the same on both.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Storage.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cstdio>
#include <cstring>
#include <exception>
#include <vector>

#include "xpuint8.h"

namespace {

using at::Tensor;

// ---------------------------------------------------------- the library
// Addresses of the loaded libxpuint8.so's entry points, in the order bind()
// receives them (_lib.py's _HOST_ENTRIES), called by the header's own types.
struct Library {
    decltype(&xpuint8_last_error) last_error;
    decltype(&xpuint8_linear_workspace_size) linear_size;
    decltype(&xpuint8_linear_packed_stream) linear;
    decltype(&xpuint8_ffn_workspace_size) ffn_size;
    decltype(&xpuint8_ffn_packed_stream) ffn;
    decltype(&xpuint8_linear_backward_int8_workspace_size) bwd_int8_size;
    decltype(&xpuint8_linear_backward_int8_stream) bwd_int8;
    decltype(&xpuint8_linear_backward_dense_workspace_size) bwd_dense_size;
    decltype(&xpuint8_linear_backward_dense_stream) bwd_dense;
    decltype(&xpuint8_linear_dx_split_workspace_size) dx_size;
    decltype(&xpuint8_linear_dx_stream) dx;
    decltype(&xpuint8_linear_dw_workspace_size) dw_size;
    decltype(&xpuint8_linear_dw_work_stream) dw;
    decltype(&xpuint8_column_sum_workspace_size) colsum_size;
    decltype(&xpuint8_column_sum_stream) colsum;
    decltype(&xpuint8_convrot_quantize_stream) quantize;
    decltype(&xpuint8_linear_acc_packed_stream) linear_acc;
    decltype(&xpuint8_linear_dx_int8_reads_packed) dx_reads_packed;
};
constexpr int kEntries = 18;
static_assert(sizeof(Library) == kEntries * sizeof(void*), "one address per entry");

Library g_lib;
PyObject* g_raw_stream = nullptr;   // device index -> current stream's handle
PyObject* g_packed = nullptr;       // the packed-weight registry (ops._PACKED)

// ----------------------------------------------------------- arguments
bool modes_active() {
    return c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           at::impl::torch_function_mode_enabled();
}

constexpr c10::DispatchKeySet kWrapped({c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper,
                                        c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                        c10::DispatchKey::Functionalize, c10::DispatchKey::Python,
                                        c10::DispatchKey::Negative, c10::DispatchKey::Conjugate,
                                        c10::DispatchKey::ZeroTensor,
                                        c10::DispatchKey::Batched});

// A plain tensor object's tensor: dense, contiguous, on a GPU, 16-byte aligned
// and not empty; null otherwise.
const Tensor* plain(PyObject* o, at::ScalarType dtype) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || t.layout() != at::kStrided || t.scalar_type() != dtype || !t.is_cuda() ||
        t.key_set().has_any(kWrapped) || !t.has_storage() || !t.is_contiguous() ||
        t.numel() == 0 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0)
        return nullptr;
    return &t;
}
// the same, one-dimensional with n values, on the device of `like`
const Tensor* vec(PyObject* o, at::ScalarType dtype, int64_t n, const Tensor& like) {
    const Tensor* t = plain(o, dtype);
    return t && t->dim() == 1 && t->numel() == n && t->device() == like.device() ? t : nullptr;
}
// an int8 [N, K] weight on the device of `like`
const Tensor* weight(PyObject* o, const Tensor& like) {
    const Tensor* t = plain(o, at::kChar);
    return t && t->dim() == 2 && t->device() == like.device() ? t : nullptr;
}

struct Bias {
    bool ok = false;
    const void* p = nullptr;
    int32_t bf16 = 0;
};
Bias bias_arg(PyObject* o, int64_t n, const Tensor& like) {
    Bias b;
    if (o == Py_None) {
        b.ok = true;
    } else if (const Tensor* t = vec(o, at::kBFloat16, n, like)) {
        b = Bias{true, t->data_ptr(), 1};
    } else if (const Tensor* t = vec(o, at::kFloat, n, like)) {
        b = Bias{true, t->data_ptr(), 0};
    }
    return b;
}

// The registry's entry of a weight (a list: weak reference to the storage,
// version, shape, packed copy, second packed form) while it is valid, borrowed;
// null without one.  The rules are ops._packed_entry's.
PyObject* packed_entry(const Tensor& w) {
    if (PyDict_GET_SIZE(g_packed) == 0 || w.is_inference() || w.storage_offset() != 0 ||
        w.size(0) % 16 != 0 || w.size(1) % 16 != 0)
        return nullptr;
    PyObject* key = PyLong_FromVoidPtr(w.storage().mutable_data());
    if (!key) throw python_error();
    PyObject* e = PyDict_GetItemWithError(g_packed, key);   // borrowed
    Py_DECREF(key);
    if (!e) {
        if (PyErr_Occurred()) throw python_error();
        return nullptr;
    }
    if (!PyList_CheckExact(e) || PyList_GET_SIZE(e) != 5) return nullptr;
    PyObject* st = PyWeakref_GetObject(PyList_GET_ITEM(e, 0));     // borrowed
    if (!st || st == Py_None ||
        THPStorage_Unpack(st).unsafeGetStorageImpl() != w.storage().unsafeGetStorageImpl())
        return nullptr;
    PyObject* shape = PyList_GET_ITEM(e, 2);
    if (PyLong_AsLongLong(PyList_GET_ITEM(e, 1)) != int64_t(w._version()) ||
        !PyTuple_CheckExact(shape) || PyTuple_GET_SIZE(shape) != 2 ||
        PyLong_AsLongLong(PyTuple_GET_ITEM(shape, 0)) != w.size(0) ||
        PyLong_AsLongLong(PyTuple_GET_ITEM(shape, 1)) != w.size(1))
        return nullptr;
    return e;
}
// entry e's packed copy (which = 3) or second form (4), undefined for none.  The
// caller holds it until its kernels are enqueued: another thread may pack the
// weight anew, or free it, as soon as the library call lets go of the GIL.
Tensor packed_form(PyObject* e, int which) {
    if (!e) return Tensor();
    PyObject* p = PyList_GET_ITEM(e, which);
    return p == Py_None ? Tensor() : THPVariable_Unpack(p);
}
const int8_t* codes(const Tensor& t) {
    return t.defined() ? static_cast<const int8_t*>(t.data_ptr()) : nullptr;
}

// ------------------------------------------------------------ the call
const void* current_stream(const Tensor& t) {
    PyObject* i = PyLong_FromLong(t.device().index());
    if (!i) throw python_error();
    PyObject* s = PyObject_CallOneArg(g_raw_stream, i);
    Py_DECREF(i);
    if (!s) throw python_error();
    const void* p = PyLong_AsVoidPtr(s);
    Py_DECREF(s);
    if (!p && PyErr_Occurred()) throw python_error();
    return p;
}
Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor& like) {
    return at::empty(sizes, at::TensorOptions().dtype(dtype).device(like.device()));
}
Tensor workspace(int64_t bytes, const Tensor& like) { return empty({bytes}, at::kByte, like); }

// RuntimeError(f"{what}: {last_error!r}"), as ops._err raises it
[[noreturn]] void fail(const char* what) {
    PyObject* msg = PyBytes_FromString(g_lib.last_error());
    if (msg) {
        PyErr_Format(PyExc_RuntimeError, "%s: %R", what, msg);
        Py_DECREF(msg);
    }
    throw python_error();
}

// The GIL released for a scope, an exception's way out of it included
struct NoGil {
    PyThreadState* s = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(s); }
};

// f() without the GIL: the allocations (as torch.empty makes them: one that
// misses the allocator's cache can wait for the device) and the library call
// (as ctypes makes it); its error, if any, raised
template <class F>
void call(const char* what, const F& f) {
    int rc;
    {
        NoGil g;
        rc = f();
    }
    if (rc != 0) fail(what);
}

// A Python-callable around f(args): C++ exceptions become Python ones
template <class F>
PyObject* guarded(Py_ssize_t nargs, Py_ssize_t want, const F& f) {
    if (nargs != want) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, nargs);
        return nullptr;
    }
    try {
        if (!g_raw_stream || !g_packed || modes_active()) Py_RETURN_NONE;
        return f();
    } catch (python_error& e) {
        // raised above with the error indicator set, or carried from torch
        if (!PyErr_Occurred()) e.restore();
        return nullptr;
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

PyObject* pair(const Tensor& a, const Tensor& b) {
    PyObject* x = THPVariable_Wrap(a);
    PyObject* y = b.defined() ? THPVariable_Wrap(b) : Py_NewRef(Py_None);
    PyObject* t = x && y ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    return t;
}

// x's leading sizes with n for the last
std::vector<int64_t> with_last(const Tensor& x, int64_t n) {
    std::vector<int64_t> s(x.sizes().begin(), x.sizes().end());
    s.back() = n;
    return s;
}

// ------------------------------------------------------------ functions
// linear(x, w8, w_scale, bias): ops.linear without activation or residual
PyObject* host_linear(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    return guarded(n_args, 4, [&]() -> PyObject* {
        const Tensor* x = plain(a[0], at::kBFloat16);
        if (!x || x->dim() < 1) Py_RETURN_NONE;
        const Tensor* w = weight(a[1], *x);
        if (!w) Py_RETURN_NONE;
        const int64_t n = w->size(0), k = w->size(1), m = x->numel() / x->size(-1);
        if (x->size(-1) != k || k % 256 != 0 || n % 16 != 0) Py_RETURN_NONE;
        const Tensor* ws = vec(a[2], at::kFloat, n, *x);
        const Bias b = bias_arg(a[3], n, *x);
        if (!ws || !b.ok) Py_RETURN_NONE;
        const int64_t need = g_lib.linear_size(m, n, k);
        if (need < 0) fail("linear");
        const Tensor packed = packed_form(packed_entry(*w), 3);
        const int8_t* p = codes(packed);
        const void* st = current_stream(*x);
        Tensor work, out;
        call("linear", [&] {
            work = workspace(need, *x);
            out = empty(with_last(*x, n), at::kBFloat16, *x);
            return g_lib.linear(st, x->data_ptr(), static_cast<const int8_t*>(w->data_ptr()), p,
                                static_cast<const float*>(ws->data_ptr()), b.p, b.bf16,
                                out.data_ptr(), m, n, k, work.data_ptr(), need);
        });
        return THPVariable_Wrap(out);
    });
}

// linear_acc(x, w8): ops.linear_acc's (int32 [M, N], fp32 [M])
PyObject* host_linear_acc(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    return guarded(n_args, 2, [&]() -> PyObject* {
        const Tensor* x = plain(a[0], at::kBFloat16);
        if (!x || x->dim() < 1) Py_RETURN_NONE;
        const Tensor* w = weight(a[1], *x);
        if (!w) Py_RETURN_NONE;
        const int64_t n = w->size(0), k = w->size(1), m = x->numel() / x->size(-1);
        if (x->size(-1) != k || k % 256 != 0 || n % 16 != 0) Py_RETURN_NONE;
        const int64_t need = g_lib.linear_size(m, n, k);
        if (need < 0) fail("linear_acc");
        const Tensor packed = packed_form(packed_entry(*w), 3);
        const int8_t* p = codes(packed);
        const void* st = current_stream(*x);
        Tensor work, acc, xs;
        call("linear_acc", [&] {
            work = workspace(need, *x);
            acc = empty({m, n}, at::kInt, *x);
            xs = empty({m}, at::kFloat, *x);
            return g_lib.linear_acc(st, x->data_ptr(), static_cast<const int8_t*>(w->data_ptr()), p,
                                    static_cast<int32_t*>(acc.data_ptr()),
                                    static_cast<float*>(xs.data_ptr()), m, n, k, work.data_ptr(),
                                    need);
        });
        return pair(acc, xs);
    });
}

// ffn(x, up_w8, up_scale, down_w8, down_scale, down_bias, activation id)
PyObject* host_ffn(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    return guarded(n_args, 7, [&]() -> PyObject* {
        const Tensor* x = plain(a[0], at::kBFloat16);
        if (!x || x->dim() < 1) Py_RETURN_NONE;
        const Tensor *up = weight(a[1], *x), *down = weight(a[3], *x);
        if (!up || !down) Py_RETURN_NONE;
        const long act = PyLong_AsLong(a[6]);
        if (act == -1 && PyErr_Occurred()) throw python_error();
        const int64_t n = up->size(0), k = up->size(1), m = x->numel() / x->size(-1);
        const bool paired = act == 3 || act == 4;
        if (!(paired || act == 5) || x->size(-1) != k || k % 256 != 0 || n % 16 != 0 ||
            (paired && n % 2 != 0))
            Py_RETURN_NONE;
        const int64_t inner = paired ? n / 2 : n;
        if (inner % 256 != 0 || down->size(0) != k || down->size(1) != inner) Py_RETURN_NONE;
        const Tensor *us = vec(a[2], at::kFloat, n, *x), *ds = vec(a[4], at::kFloat, k, *x);
        const Bias b = bias_arg(a[5], k, *x);
        if (!us || !ds || !b.ok) Py_RETURN_NONE;
        const int64_t need = g_lib.ffn_size(m, inner, k, int32_t(act));
        if (need < 0) fail("ffn");
        const Tensor up_packed = packed_form(packed_entry(*up), 3),
                     down_packed = packed_form(packed_entry(*down), 3);
        const int8_t *up_p = codes(up_packed), *down_p = codes(down_packed);
        const void* st = current_stream(*x);
        Tensor work, out;
        call("ffn", [&] {
            work = workspace(need, *x);
            out = empty(x->sizes(), at::kBFloat16, *x);
            return g_lib.ffn(st, x->data_ptr(), static_cast<const int8_t*>(up->data_ptr()), up_p,
                             static_cast<const float*>(us->data_ptr()),
                             static_cast<const int8_t*>(down->data_ptr()), down_p,
                             static_cast<const float*>(ds->data_ptr()), b.p, b.bf16, out.data_ptr(),
                             m, inner, k, int32_t(act), work.data_ptr(), need);
        });
        return THPVariable_Wrap(out);
    });
}

// backward(dy, w8, w_scale, want_dbias, dbias_fp32, dense): ops._linear_backward's
// (dx, dbias or None).  The int8 mode of a weight whose second packed form this
// product reads and is still to be made goes through Python, which makes it.
PyObject* host_backward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    return guarded(n_args, 6, [&]() -> PyObject* {
        const Tensor* dy = plain(a[0], at::kBFloat16);
        if (!dy || dy->dim() != 2) Py_RETURN_NONE;
        const Tensor* w = weight(a[1], *dy);
        if (!w) Py_RETURN_NONE;
        const int64_t m = dy->size(0), n = w->size(0), k = w->size(1);
        if (dy->size(1) != n || n % 16 != 0 || k % 256 != 0) Py_RETURN_NONE;
        const Tensor* ws = vec(a[2], at::kFloat, n, *dy);
        if (!ws) Py_RETURN_NONE;
        const int want = PyObject_IsTrue(a[3]), f32 = PyObject_IsTrue(a[4]),
                  dense = PyObject_IsTrue(a[5]);
        if (want < 0 || f32 < 0 || dense < 0) throw python_error();
        const char* what = dense ? "linear_dx" : "linear_dx_int8";
        Tensor packed_nn;
        if (!dense) {
            PyObject* e = packed_entry(*w);
            packed_nn = packed_form(e, 4);
            if (e && !packed_nn.defined() && g_lib.dx_reads_packed(m, n, k) == 1) Py_RETURN_NONE;
        }
        const int8_t* nn = codes(packed_nn);
        const int64_t need = (dense ? g_lib.bwd_dense_size : g_lib.bwd_int8_size)(m, n, k);
        if (need < 0) fail(what);
        const int8_t* wp = static_cast<const int8_t*>(w->data_ptr());
        const float* wsp = static_cast<const float*>(ws->data_ptr());
        const void* st = current_stream(*dy);
        Tensor work, dx, db;
        call(what, [&] {
            work = workspace(need, *dy);
            dx = empty({m, k}, at::kBFloat16, *dy);
            if (want) db = empty({n}, f32 ? at::kFloat : at::kBFloat16, *dy);
            void* dbp = want ? db.data_ptr() : nullptr;
            return dense ? g_lib.bwd_dense(st, dy->data_ptr(), wp, wsp, dx.data_ptr(), dbp,
                                           want && f32, m, n, k, work.data_ptr(), need)
                         : g_lib.bwd_int8(st, dy->data_ptr(), wsp, wp, nn, dx.data_ptr(), dbp,
                                          want && f32, m, n, k, work.data_ptr(), need);
        });
        return pair(dx, db);
    });
}

// linear_dx(dy, w): dy [.., N] @ w [N, K], both bf16
PyObject* host_linear_dx(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    return guarded(n_args, 2, [&]() -> PyObject* {
        const Tensor *dy = plain(a[0], at::kBFloat16), *w = plain(a[1], at::kBFloat16);
        if (!dy || !w || dy->dim() < 1 || w->dim() != 2 || w->device() != dy->device())
            Py_RETURN_NONE;
        const int64_t n = w->size(0), k = w->size(1), m = dy->numel() / dy->size(-1);
        if (dy->size(-1) != n || n % 16 != 0 || k % 16 != 0) Py_RETURN_NONE;
        const int64_t need = g_lib.dx_size(m, n, k);
        if (need < 0) fail("linear_dx");
        const void* st = current_stream(*dy);
        Tensor work, dx;
        call("linear_dx", [&] {
            if (need > 0) work = workspace(need, *dy);
            dx = empty(with_last(*dy, k), at::kBFloat16, *dy);
            return g_lib.dx(st, dy->data_ptr(), w->data_ptr(), dx.data_ptr(), m, n, k,
                            need > 0 ? work.data_ptr() : nullptr, need);
        });
        return THPVariable_Wrap(dx);
    });
}

// linear_dw(dy, x): dy [M, N]^T @ x [M, K], both bf16
PyObject* host_linear_dw(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    return guarded(n_args, 2, [&]() -> PyObject* {
        const Tensor *dy = plain(a[0], at::kBFloat16), *x = plain(a[1], at::kBFloat16);
        if (!dy || !x || dy->dim() != 2 || x->dim() != 2 || x->device() != dy->device() ||
            dy->size(0) != x->size(0))
            Py_RETURN_NONE;
        const int64_t m = dy->size(0), n = dy->size(1), k = x->size(1);
        if (n % 16 != 0 || k % 16 != 0) Py_RETURN_NONE;
        const int64_t need = g_lib.dw_size(m, n, k);
        if (need < 0) fail("linear_dw");
        const void* st = current_stream(*dy);
        Tensor work, dw;
        call("linear_dw", [&] {
            if (need > 0) work = workspace(need, *dy);
            dw = empty({n, k}, at::kBFloat16, *dy);
            return g_lib.dw(st, dy->data_ptr(), x->data_ptr(), dw.data_ptr(), m, n, k,
                            need > 0 ? work.data_ptr() : nullptr, need);
        });
        return THPVariable_Wrap(dw);
    });
}

// column_sum(dy): the column sums of a bf16 [M, N]
PyObject* host_column_sum(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    return guarded(n_args, 1, [&]() -> PyObject* {
        const Tensor* dy = plain(a[0], at::kBFloat16);
        if (!dy || dy->dim() != 2 || dy->size(1) % 16 != 0) Py_RETURN_NONE;
        const int64_t m = dy->size(0), n = dy->size(1), need = g_lib.colsum_size(m, n);
        if (need < 0) fail("column_sum");
        const void* st = current_stream(*dy);
        Tensor work, out;
        call("column_sum", [&] {
            work = workspace(std::max<int64_t>(need, 16), *dy);
            out = empty({n}, at::kBFloat16, *dy);
            return g_lib.colsum(st, dy->data_ptr(), out.data_ptr(), m, n, work.data_ptr(), need);
        });
        return THPVariable_Wrap(out);
    });
}

// quantize(x): ops.quantize's (int8 [.., K], fp32 [..])
PyObject* host_quantize(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    return guarded(n_args, 1, [&]() -> PyObject* {
        const Tensor* x = plain(a[0], at::kBFloat16);
        if (!x || x->dim() < 1) Py_RETURN_NONE;
        const int64_t k = x->size(-1), m = x->numel() / k;
        const void* st = current_stream(*x);
        Tensor q, s;
        call("quantize", [&] {
            q = empty(x->sizes(), at::kChar, *x);
            s = empty(x->sizes().slice(0, x->dim() - 1), at::kFloat, *x);
            return g_lib.quantize(st, x->data_ptr(), static_cast<int8_t*>(q.data_ptr()),
                                  static_cast<float*>(s.data_ptr()), m, k);
        });
        return pair(q, s);
    });
}

// bind(addresses, raw_stream, packed): the library's entry points in Library's
// order, the current-stream accessor and the packed-weight registry
PyObject* host_bind(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    if (n_args != 3 || !PyTuple_CheckExact(a[0]) || PyTuple_GET_SIZE(a[0]) != kEntries ||
        !PyCallable_Check(a[1]) || !PyDict_CheckExact(a[2])) {
        PyErr_SetString(PyExc_TypeError, "bind(tuple of addresses, callable, dict)");
        return nullptr;
    }
    std::array<void*, kEntries> p;
    for (int i = 0; i < kEntries; ++i) {
        p[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(a[0], i));
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
            return nullptr;
        }
    }
    std::memcpy(static_cast<void*>(&g_lib), p.data(), sizeof(g_lib));
    Py_XSETREF(g_raw_stream, Py_NewRef(a[1]));
    Py_XSETREF(g_packed, Py_NewRef(a[2]));
    Py_RETURN_NONE;
}

#define XPU_HOST(name, fn) \
    {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(fn)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {XPU_HOST("bind", host_bind),
                          XPU_HOST("linear", host_linear),
                          XPU_HOST("linear_acc", host_linear_acc),
                          XPU_HOST("ffn", host_ffn),
                          XPU_HOST("backward", host_backward),
                          XPU_HOST("linear_dx", host_linear_dx),
                          XPU_HOST("linear_dw", host_linear_dw),
                          XPU_HOST("column_sum", host_column_sum),
                          XPU_HOST("quantize", host_quantize),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host",
                       "The int8 API's hot calls in native code (see host_ops.cpp).", -1, kMethods};

// Tensors are read by the layout that torch's headers gave at build time, and
// another build of torch can export the same symbols over another layout: the
// module loads only into the Python and the torch (version and commit) that the
// Makefile found, XPU_BUILT_FOR = "3.10/2.10.0+rocm7.0/<commit>", and raises
// ImportError elsewhere.
bool built_for_this() {
    int major = 0, minor = 0;
    std::sscanf(Py_GetVersion(), "%d.%d", &major, &minor);
    PyObject* v = PyImport_ImportModule("torch.version");
    PyObject* version = v ? PyObject_GetAttrString(v, "__version__") : nullptr;
    PyObject* commit = version ? PyObject_GetAttrString(v, "git_version") : nullptr;
    PyObject* now = commit ? PyUnicode_FromFormat("%d.%d/%S/%S", major, minor, version, commit)
                           : nullptr;
    const bool ok = now && PyUnicode_CompareWithASCIIString(now, XPU_BUILT_FOR) == 0;
    if (!ok) {
        PyErr_Clear();
        PyErr_Format(PyExc_ImportError, "_host.so was built for " XPU_BUILT_FOR ", not %S",
                     now ? now : Py_None);
    }
    Py_XDECREF(now);
    Py_XDECREF(commit);
    Py_XDECREF(version);
    Py_XDECREF(v);
    return ok;
}

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    if (!built_for_this()) return nullptr;
    return PyModule_Create(&kModule);
}
