// The host side of one operator call in native code: allocate the outputs, look up the current stream, call the C ABI of
// libthnorm.so (TritonHub/_host.so).
//
// Each function takes what the Python wrapper of the same name takes (TritonHub/*/_launch.py) and does what that wrapper
// does for the ordinary call: plain tensors of a supported type, contiguous, not empty, on the current device.  For
// anything else it returns None and the wrapper goes its general way (strides, empty tensors, other devices, tensor
// subclasses, mixed types, every error message).
//
// Small calls are bound by this work: a forward + backward of a float32 LayerNorm over 2 x 100 x 128, whose kernels take
// 14 us, took 118 us with the wrappers in Python (three allocations, a workspace look-up under a lock and up to 18
// converted arguments per direction) and takes 80 with these; an RMSNorm of 64 x 4096 without gradients 13.8 -> 10.4; a
// float16 LayerNorm of 8192 x 6000, whose kernels take 92 us, 118 -> 87; a bfloat16 softmax of 768 x 197 x 197 74 -> 55.
// Of what is left of the first, an empty autograd function takes 37 us (backward 32) and the kernels 14; the rest, not measured
// apart, is the body of the Python autograd function (its saved tensors, the call of the wrapper) and these calls.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/SavedTensorHooks.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "thn_dropout_mask.h"
#include "thnorm.h"

namespace {

constexpr int64_t kMaxNormRowBytes = 65536;

int type_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return THN_F32;
        case at::kHalf: return THN_F16;
        case at::kBFloat16: return THN_BF16;
        case at::kDouble: return THN_F64;
        default: return -1;
    }
}

// A tensor (or parameter, no subclass of either) that the C ABI can take as it is: dense on the current device.
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.dim() < 1 || t.numel() == 0 || !t.is_contiguous()) return nullptr;
    if (type_code(t) < 0 || t.get_device() != c10::hip::current_device()) return nullptr;
    return &t;
}

// An optional parameter of n elements: `out` is null for None; false where the general way has to look at it.
bool plain_param(PyObject* o, int64_t n, const at::Tensor** out) {
    *out = nullptr;
    if (o == Py_None) return true;
    *out = plain(o);
    return *out != nullptr && (*out)->dim() == 1 && (*out)->size(0) == n;
}

void* address(const at::Tensor* t) { return t == nullptr ? nullptr : t->data_ptr(); }
void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// The C ABI runs without the interpreter's lock, as a ctypes call does.  An exception on its way out (an allocation or a mutex
// of the library's caches) finds the lock held again: HANDLE_TH_ERRORS turns it into a Python error.
struct Unlocked {
    PyThreadState* const state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename Fn> int unlocked(Fn&& fn) {
    const Unlocked here;
    return fn();
}

PyObject* failed(int status) {
    return PyErr_Format(PyExc_RuntimeError, "libthnorm: %s (status %d)", thn_strerror(status), status);
}

// Moves the tensors into a tuple; an undefined one becomes None.
template <size_t N> PyObject* as_tuple(const at::Tensor (&tensors)[N]) {
    PyObject* result = PyTuple_New(N);
    if (result == nullptr) return nullptr;
    for (size_t i = 0; i < N; ++i) {
        PyObject* o = tensors[i].defined() ? THPVariable_Wrap(tensors[i]) : Py_NewRef(Py_None);
        if (o == nullptr) {
            Py_DECREF(result);
            return nullptr;
        }
        PyTuple_SET_ITEM(result, i, o);
    }
    return result;
}

// Numbers that do not convert (a tensor that needs its own conversion, an overflow) are the general way's as well.
bool number(PyObject* o, double* v) {
    *v = PyFloat_AsDouble(o);
    if (*v == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}
bool whole(PyObject* o, long long* v) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    *v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}
bool wrong_count(Py_ssize_t got, Py_ssize_t want) {
    if (got == want) return false;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, got);
    return true;
}

// norm_fwd(x, weight, bias, eps, layernorm, act, x_flags) -> (out, mean or None, rstd)
PyObject* norm_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 7)) return nullptr;
    const at::Tensor* x = plain(args[0]);
    double eps;
    long long act, flags;
    if (x == nullptr || !number(args[3], &eps) || !whole(args[5], &act) || !whole(args[6], &flags)) Py_RETURN_NONE;
    const int64_t n = x->size(-1), m = x->numel() / n;
    const at::Tensor *w, *b;
    if (n * x->element_size() > kMaxNormRowBytes || !plain_param(args[1], n, &w) || !plain_param(args[2], n, &b)) Py_RETURN_NONE;
    if (w != nullptr && b != nullptr && w->scalar_type() != b->scalar_type()) Py_RETURN_NONE;
    const bool layernorm = PyObject_IsTrue(args[4]) == 1;
    const at::Tensor* param = w != nullptr ? w : b;
    const int x_code = type_code(*x) | static_cast<int>(flags), w_code = param != nullptr ? type_code(*param) : type_code(*x);
    const auto statistics = x->options().dtype(at::kFloat);
    at::Tensor results[3] = {at::empty_like(*x), layernorm ? at::empty({m}, statistics) : at::Tensor(), at::empty({m}, statistics)};
    void* xp = x->data_ptr();
    void* yp = results[0].data_ptr();
    float* mean = layernorm ? results[1].data_ptr<float>() : nullptr;
    float* rstd = results[2].data_ptr<float>();
    void *wp = address(w), *bp = address(b), *stream = stream_of(*x);
    const int status = unlocked([&] {
        if (act < 0) return thn_norm_fwd(xp, n, yp, n, wp, bp, mean, rstd, m, n, static_cast<float>(eps), x_code, w_code, stream);
        return thn_norm_act_fwd(xp, n, yp, n, wp, bp, mean, rstd, m, n, static_cast<float>(eps), static_cast<int>(act), x_code, w_code, stream);
    });
    if (status != THN_OK) return failed(status);
    return as_tuple(results);
    END_HANDLE_TH_ERRORS
}

// norm_bwd(x, dout, weight, bias, mean, rstd, layernorm, act, need_dw, need_db) -> (dx, dw or None, db or None).  The partial
// sums' workspace comes from torch's allocator on every call: it is reused in the order of the stream it is allocated on,
// by a captured graph from the graph's own pool, so no lock has to keep two calls apart.
PyObject* norm_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 10)) return nullptr;
    const at::Tensor *x = plain(args[0]), *g = plain(args[1]), *rstd = plain(args[5]);
    const bool layernorm = PyObject_IsTrue(args[6]) == 1;
    const at::Tensor* mean = layernorm ? plain(args[4]) : nullptr;
    long long act;
    if (x == nullptr || g == nullptr || rstd == nullptr || (layernorm && mean == nullptr) || !whole(args[7], &act)) Py_RETURN_NONE;
    const int64_t n = x->size(-1), m = x->numel() / n;
    const at::Tensor *w, *b;
    if (n * x->element_size() > kMaxNormRowBytes || !plain_param(args[2], n, &w) || !plain_param(args[3], n, &b)) Py_RETURN_NONE;
    if (!layernorm) b = nullptr;
    if (b != nullptr && (w == nullptr || w->scalar_type() != b->scalar_type())) Py_RETURN_NONE;
    if (g->size(-1) != n || g->numel() != x->numel() || g->scalar_type() != x->scalar_type()) Py_RETURN_NONE;
    if (rstd->scalar_type() != at::kFloat || rstd->numel() != m) Py_RETURN_NONE;
    if (layernorm && (mean->scalar_type() != at::kFloat || mean->numel() != m)) Py_RETURN_NONE;
    const int x_code = type_code(*x), w_code = w != nullptr ? type_code(*w) : x_code;
    const bool want_dw = w != nullptr && PyObject_IsTrue(args[8]) == 1, want_db = b != nullptr && PyObject_IsTrue(args[9]) == 1;
    const int64_t bytes = act < 0 ? thn_norm_bwd_workspace_bytes(m, n, want_dw, want_db, x_code)
                                  : thn_norm_act_bwd_workspace_bytes(m, n, want_dw, want_db, static_cast<int>(act), x_code);
    if (bytes < 0) return failed(static_cast<int>(bytes));
    at::Tensor results[3] = {at::empty_like(*x), want_dw ? at::empty_like(*w) : at::Tensor(), want_db ? at::empty_like(*b) : at::Tensor()};
    const at::Tensor workspace = bytes > 0 ? at::empty({bytes}, x->options().dtype(at::kByte)) : at::Tensor();
    void *xp = x->data_ptr(), *gp = g->data_ptr(), *dxp = results[0].data_ptr(), *wp = address(w), *bp = address(b);
    const float *mean_p = layernorm ? mean->data_ptr<float>() : nullptr, *rstd_p = rstd->data_ptr<float>();
    void *dwp = want_dw ? results[1].data_ptr() : nullptr, *dbp = want_db ? results[2].data_ptr() : nullptr;
    void *ws = bytes > 0 ? workspace.data_ptr() : nullptr, *stream = stream_of(*x);
    const int status = unlocked([&] {
        if (act < 0) return thn_norm_bwd(xp, n, gp, n, dxp, n, wp, mean_p, rstd_p, dwp, dbp, ws, bytes, m, n, x_code, w_code, stream);
        return thn_norm_act_bwd(xp, n, gp, n, dxp, n, wp, bp, mean_p, rstd_p, dwp, dbp, ws, bytes, m, n, static_cast<int>(act), x_code, w_code, stream);
    });
    if (status != THN_OK) return failed(status);
    return as_tuple(results);
    END_HANDLE_TH_ERRORS
}

// Both tensors of a backward can be passed as they are and describe the same rows.
bool plain_pair(PyObject* saved, PyObject* upstream, const at::Tensor** s, const at::Tensor** g) {
    *s = plain(saved);
    *g = plain(upstream);
    return *s != nullptr && *g != nullptr && (*g)->size(-1) == (*s)->size(-1) && (*g)->numel() == (*s)->numel() &&
           (*g)->scalar_type() == (*s)->scalar_type();
}

// softmax_fwd(x, kind) -> out
PyObject* softmax_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 2)) return nullptr;
    const at::Tensor* x = plain(args[0]);
    long long kind;
    if (x == nullptr || !whole(args[1], &kind)) Py_RETURN_NONE;
    const at::Tensor out = at::empty_like(*x);
    const int64_t n = x->size(-1), m = x->numel() / n;
    void *xp = x->data_ptr(), *yp = out.data_ptr(), *stream = stream_of(*x);
    const int code = type_code(*x);
    const int status = unlocked([&] { return thn_softmax_fwd(xp, n, yp, n, m, n, static_cast<int>(kind), code, stream); });
    if (status != THN_OK) return failed(status);
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// softmax_bwd(y, dout, kind) -> dx
PyObject* softmax_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 3)) return nullptr;
    const at::Tensor *y, *g;
    long long kind;
    if (!plain_pair(args[0], args[1], &y, &g) || !whole(args[2], &kind)) Py_RETURN_NONE;
    const at::Tensor dx = at::empty_like(*y);
    const int64_t n = y->size(-1), m = y->numel() / n;
    void *yp = y->data_ptr(), *gp = g->data_ptr(), *dxp = dx.data_ptr(), *stream = stream_of(*y);
    const int code = type_code(*y);
    const int status = unlocked([&] { return thn_softmax_bwd(yp, n, gp, n, dxp, n, m, n, static_cast<int>(kind), code, stream); });
    if (status != THN_OK) return failed(status);
    return THPVariable_Wrap(dx);
    END_HANDLE_TH_ERRORS
}

// act_fwd(x, act, param0, param1) -> out
PyObject* act_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 4)) return nullptr;
    const at::Tensor* x = plain(args[0]);
    long long act;
    double p0, p1;
    if (x == nullptr || !whole(args[1], &act) || !number(args[2], &p0) || !number(args[3], &p1)) Py_RETURN_NONE;
    const at::Tensor out = at::empty_like(*x);
    const int64_t n = x->size(-1), m = x->numel() / n;
    void *xp = x->data_ptr(), *yp = out.data_ptr(), *stream = stream_of(*x);
    const int code = type_code(*x);
    const int status = unlocked([&] {
        return thn_act_fwd(xp, n, yp, n, m, n, static_cast<int>(act), static_cast<float>(p0), static_cast<float>(p1), code, stream);
    });
    if (status != THN_OK) return failed(status);
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// act_bwd(saved, dout, act, param0, param1) -> dx
PyObject* act_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 5)) return nullptr;
    const at::Tensor *s, *g;
    long long act;
    double p0, p1;
    if (!plain_pair(args[0], args[1], &s, &g) || !whole(args[2], &act) || !number(args[3], &p0) || !number(args[4], &p1)) Py_RETURN_NONE;
    const at::Tensor dx = at::empty_like(*s);
    const int64_t n = s->size(-1), m = s->numel() / n;
    void *sp = s->data_ptr(), *gp = g->data_ptr(), *dxp = dx.data_ptr(), *stream = stream_of(*s);
    const int code = type_code(*s);
    const int status = unlocked([&] {
        return thn_act_bwd(sp, n, gp, n, dxp, n, m, n, static_cast<int>(act), static_cast<float>(p0), static_cast<float>(p1), code, stream);
    });
    if (status != THN_OK) return failed(status);
    return THPVariable_Wrap(dx);
    END_HANDLE_TH_ERRORS
}

constexpr int64_t kMaskTo = int64_t{1} << 32;        // the masked kernels take offsets of 32 bits

// dropout_fwd(x, p, seed, keep) -> (out, mask or None), for 0 < p < 1 (in float32, as the kernels compare); keep: the decisions
// are wanted for a backward (one byte per 16 bytes of input, in 32-bit words).  Under saved-tensor hooks (offloading, a
// non-reentrant checkpoint) none are kept: the hooks would not see the mask, and it would stay where they are to free memory.
PyObject* dropout_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 4)) return nullptr;
    const at::Tensor* x = plain(args[0]);
    double p;
    long long seed;
    if (x == nullptr || !number(args[1], &p) || !(p > 0.0 && static_cast<float>(p) < 1.0f) || !whole(args[2], &seed)) Py_RETURN_NONE;
    const int64_t n = x->numel();
    const bool keep = PyObject_IsTrue(args[3]) == 1 && n < kMaskTo && at::SavedTensorDefaultHooks::get_tls_state().stack.empty();
    // (contiguous strides also for dimensions of one element, whose strides empty_like would take over from x)
    at::Tensor results[2] = {at::empty_like(*x, at::MemoryFormat::Contiguous),
                             keep ? at::empty({thn::dropout_mask_words(n, static_cast<int>(x->element_size()))}, x->options().dtype(at::kInt)) : at::Tensor()};
    void *xp = x->data_ptr(), *yp = results[0].data_ptr(), *stream = stream_of(*x);
    uint32_t* mask = keep ? reinterpret_cast<uint32_t*>(results[1].data_ptr<int32_t>()) : nullptr;
    const int code = type_code(*x);
    const int status = unlocked([&] {
        if (keep) return thn::dropout_keep_mask(xp, yp, mask, n, static_cast<float>(p), static_cast<uint64_t>(seed), code, stream);
        return thn_dropout(xp, yp, n, 0, static_cast<float>(p), static_cast<uint64_t>(seed), code, stream);
    });
    if (status != THN_OK) return failed(status);
    return as_tuple(results);
    END_HANDLE_TH_ERRORS
}

// dropout_bwd(dout, p, seed, mask or None) -> dx; a mask of another size belongs to another type of storage
PyObject* dropout_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 4)) return nullptr;
    const at::Tensor* g = plain(args[0]);
    double p;
    long long seed;
    if (g == nullptr || !number(args[1], &p) || !(p > 0.0 && static_cast<float>(p) < 1.0f) || !whole(args[2], &seed)) Py_RETURN_NONE;
    const int64_t n = g->numel();
    const uint32_t* mask = nullptr;
    if (args[3] != Py_None) {
        if (!THPVariable_CheckExact(args[3])) Py_RETURN_NONE;
        const at::Tensor& t = THPVariable_Unpack(args[3]);
        if (!t.defined() || t.device() != g->device() || t.scalar_type() != at::kInt || !t.is_contiguous() ||
            t.numel() != thn::dropout_mask_words(n, static_cast<int>(g->element_size()))) {
            Py_RETURN_NONE;
        }
        mask = reinterpret_cast<const uint32_t*>(t.data_ptr<int32_t>());
    }
    const at::Tensor dx = at::empty_like(*g, at::MemoryFormat::Contiguous);
    void *gp = g->data_ptr(), *dxp = dx.data_ptr(), *stream = stream_of(*g);
    const int code = type_code(*g);
    const int status = unlocked([&] {
        if (mask != nullptr) return thn::dropout_from_mask(gp, dxp, mask, n, static_cast<float>(p), static_cast<uint64_t>(seed), code, stream);
        return thn_dropout(gp, dxp, n, 0, static_cast<float>(p), static_cast<uint64_t>(seed), code, stream);
    });
    if (status != THN_OK) return failed(status);
    return THPVariable_Wrap(dx);
    END_HANDLE_TH_ERRORS
}

#define THN_METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(NAME)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {THN_METHOD(norm_fwd),    THN_METHOD(norm_bwd), THN_METHOD(softmax_fwd), THN_METHOD(softmax_bwd),
                         THN_METHOD(act_fwd),     THN_METHOD(act_bwd),
                         THN_METHOD(dropout_fwd), THN_METHOD(dropout_bwd), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Host side of the operator calls in native code.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
