// The host side of one operator call in native code: allocate the outputs, look up the current stream, call the C ABI of
// libthnorm.so (TritonHub/_host.so).
//
// Each function takes what the Python wrapper of the same name takes (TritonHub/*/_launch.py) and does what that wrapper
// does for the ordinary call: plain tensors of a supported type, contiguous, not empty, on the current device.  For
// anything else it returns None and the wrapper goes its general way (strides, empty tensors, other devices, tensor
// subclasses, mixed types, every error message).
//
// Small calls are bound by this work.  us per forward + backward with the operator in Python (wrapper and autograd Function) -> the wrapper
// native -> the Function native too (below, "The autograd Functions"): float32 LayerNorm over 2 x 100 x 128, whose kernels take 14,
// 118 -> 88 -> 73; float32 normalize of the same 98 -> 98 -> 53; bfloat16 softmax of 768 x 197 x 197 74 -> 55 -> 50; an RMSNorm of
// 64 x 4096 without gradients 13.8 -> 10.4 -> 7.9.  An x * 2 of torch's with its backward takes 43 there: the autograd engine
// and three launches.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/autograd/python_variable.h>

#include <utility>
#include <vector>

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

// What became of a call: made, left to the general way, or refused by the library (a Python error is set).
enum class Call { kMade, kGeneral, kFailed };
Call outcome(int status) {
    if (status == THN_OK) return Call::kMade;
    failed(status);
    return Call::kFailed;
}

// results: out, mean or undefined, rstd; `apart` false: the statistics are not wanted and lie in one allocation (an allocation takes 1.2 us)
Call norm_forward(PyObject* input, PyObject* weight, PyObject* bias, PyObject* eps_number, bool layernorm, long long act, int flags, bool apart, at::Tensor (&results)[3]) {
    const at::Tensor* x = plain(input);
    double eps;
    if (x == nullptr || !number(eps_number, &eps)) return Call::kGeneral;
    const int64_t n = x->size(-1), m = x->numel() / n;
    const at::Tensor *w, *b;
    if (n * x->element_size() > kMaxNormRowBytes || !plain_param(weight, n, &w) || !plain_param(bias, n, &b)) return Call::kGeneral;
    if (w != nullptr && b != nullptr && w->scalar_type() != b->scalar_type()) return Call::kGeneral;
    const at::Tensor* param = w != nullptr ? w : b;
    const int x_code = type_code(*x) | flags, w_code = param != nullptr ? type_code(*param) : type_code(*x);
    const auto statistics = x->options().dtype(at::kFloat);
    results[0] = at::empty_like(*x);
    if (layernorm && apart) results[1] = at::empty({m}, statistics);
    results[2] = at::empty({layernorm && !apart ? 2 * m : m}, statistics);
    void* xp = x->data_ptr();
    void* yp = results[0].data_ptr();
    float* rstd = results[2].data_ptr<float>();
    float* mean = !layernorm ? nullptr : apart ? results[1].data_ptr<float>() : rstd + m;
    void *wp = address(w), *bp = address(b), *stream = stream_of(*x);
    return outcome(unlocked([&] {
        if (act < 0) return thn_norm_fwd(xp, n, yp, n, wp, bp, mean, rstd, m, n, static_cast<float>(eps), x_code, w_code, stream);
        return thn_norm_act_fwd(xp, n, yp, n, wp, bp, mean, rstd, m, n, static_cast<float>(eps), static_cast<int>(act), x_code, w_code, stream);
    }));
}

// norm_fwd(x, weight, bias, eps, layernorm, act, x_flags) -> (out, mean or None, rstd)
PyObject* norm_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 7)) return nullptr;
    long long act, flags;
    if (!whole(args[5], &act) || !whole(args[6], &flags)) Py_RETURN_NONE;
    at::Tensor results[3];
    const Call call = norm_forward(args[0], args[1], args[2], args[3], PyObject_IsTrue(args[4]) == 1, act, static_cast<int>(flags), true, results);
    if (call == Call::kGeneral) Py_RETURN_NONE;
    return call == Call::kMade ? as_tuple(results) : nullptr;
    END_HANDLE_TH_ERRORS
}

// results: dx, dw or undefined, db or undefined.  The partial sums' workspace comes from torch's allocator on every call: it is
// reused in the order of the stream it is allocated on, by a captured graph from the graph's own pool, so no lock has to keep
// two calls apart.
Call norm_backward(PyObject* input, PyObject* d_out, PyObject* weight, PyObject* bias, PyObject* saved_mean, PyObject* saved_rstd, bool layernorm, long long act,
                   bool need_dw, bool need_db, at::Tensor (&results)[3]) {
    const at::Tensor *x = plain(input), *g = plain(d_out), *rstd = plain(saved_rstd);
    const at::Tensor* mean = layernorm ? plain(saved_mean) : nullptr;
    if (x == nullptr || g == nullptr || rstd == nullptr || (layernorm && mean == nullptr)) return Call::kGeneral;
    const int64_t n = x->size(-1), m = x->numel() / n;
    const at::Tensor *w, *b;
    if (n * x->element_size() > kMaxNormRowBytes || !plain_param(weight, n, &w) || !plain_param(bias, n, &b)) return Call::kGeneral;
    if (!layernorm) b = nullptr;
    if (b != nullptr && (w == nullptr || w->scalar_type() != b->scalar_type())) return Call::kGeneral;
    if (g->size(-1) != n || g->numel() != x->numel() || g->scalar_type() != x->scalar_type()) return Call::kGeneral;
    if (rstd->scalar_type() != at::kFloat || rstd->numel() != m) return Call::kGeneral;
    if (layernorm && (mean->scalar_type() != at::kFloat || mean->numel() != m)) return Call::kGeneral;
    const int x_code = type_code(*x), w_code = w != nullptr ? type_code(*w) : x_code;
    const bool want_dw = w != nullptr && need_dw, want_db = b != nullptr && need_db;
    const int64_t bytes = act < 0 ? thn_norm_bwd_workspace_bytes(m, n, want_dw, want_db, x_code)
                                  : thn_norm_act_bwd_workspace_bytes(m, n, want_dw, want_db, static_cast<int>(act), x_code);
    if (bytes < 0) return outcome(static_cast<int>(bytes));
    results[0] = at::empty_like(*x);
    if (want_dw) results[1] = at::empty_like(*w);
    if (want_db) results[2] = at::empty_like(*b);
    const at::Tensor workspace = bytes > 0 ? at::empty({bytes}, x->options().dtype(at::kByte)) : at::Tensor();
    void *xp = x->data_ptr(), *gp = g->data_ptr(), *dxp = results[0].data_ptr(), *wp = address(w), *bp = address(b);
    const float *mean_p = layernorm ? mean->data_ptr<float>() : nullptr, *rstd_p = rstd->data_ptr<float>();
    void *dwp = want_dw ? results[1].data_ptr() : nullptr, *dbp = want_db ? results[2].data_ptr() : nullptr;
    void *ws = bytes > 0 ? workspace.data_ptr() : nullptr, *stream = stream_of(*x);
    return outcome(unlocked([&] {
        if (act < 0) return thn_norm_bwd(xp, n, gp, n, dxp, n, wp, mean_p, rstd_p, dwp, dbp, ws, bytes, m, n, x_code, w_code, stream);
        return thn_norm_act_bwd(xp, n, gp, n, dxp, n, wp, bp, mean_p, rstd_p, dwp, dbp, ws, bytes, m, n, static_cast<int>(act), x_code, w_code, stream);
    }));
}

// norm_bwd(x, dout, weight, bias, mean, rstd, layernorm, act, need_dw, need_db) -> (dx, dw or None, db or None)
PyObject* norm_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 10)) return nullptr;
    long long act;
    if (!whole(args[7], &act)) Py_RETURN_NONE;
    at::Tensor results[3];
    const Call call = norm_backward(args[0], args[1], args[2], args[3], args[4], args[5], PyObject_IsTrue(args[6]) == 1, act, PyObject_IsTrue(args[8]) == 1,
                                    PyObject_IsTrue(args[9]) == 1, results);
    if (call == Call::kGeneral) Py_RETURN_NONE;
    return call == Call::kMade ? as_tuple(results) : nullptr;
    END_HANDLE_TH_ERRORS
}

// Both tensors of a backward can be passed as they are and describe the same rows.
bool plain_pair(PyObject* saved, PyObject* upstream, const at::Tensor** s, const at::Tensor** g) {
    *s = plain(saved);
    *g = plain(upstream);
    return *s != nullptr && *g != nullptr && (*g)->size(-1) == (*s)->size(-1) && (*g)->numel() == (*s)->numel() &&
           (*g)->scalar_type() == (*s)->scalar_type();
}

Call softmax_forward(PyObject* input, int kind, at::Tensor& out) {
    const at::Tensor* x = plain(input);
    if (x == nullptr) return Call::kGeneral;
    out = at::empty_like(*x);
    const int64_t n = x->size(-1), m = x->numel() / n;
    void *xp = x->data_ptr(), *yp = out.data_ptr(), *stream = stream_of(*x);
    const int code = type_code(*x);
    return outcome(unlocked([&] { return thn_softmax_fwd(xp, n, yp, n, m, n, kind, code, stream); }));
}

Call softmax_backward(PyObject* saved, PyObject* d_out, int kind, at::Tensor& dx) {
    const at::Tensor *y, *g;
    if (!plain_pair(saved, d_out, &y, &g)) return Call::kGeneral;
    dx = at::empty_like(*y);
    const int64_t n = y->size(-1), m = y->numel() / n;
    void *yp = y->data_ptr(), *gp = g->data_ptr(), *dxp = dx.data_ptr(), *stream = stream_of(*y);
    const int code = type_code(*y);
    return outcome(unlocked([&] { return thn_softmax_bwd(yp, n, gp, n, dxp, n, m, n, kind, code, stream); }));
}

Call act_forward(PyObject* input, int act, double p0, double p1, at::Tensor& out) {
    const at::Tensor* x = plain(input);
    if (x == nullptr) return Call::kGeneral;
    out = at::empty_like(*x);
    const int64_t n = x->size(-1), m = x->numel() / n;
    void *xp = x->data_ptr(), *yp = out.data_ptr(), *stream = stream_of(*x);
    const int code = type_code(*x);
    return outcome(unlocked([&] { return thn_act_fwd(xp, n, yp, n, m, n, act, static_cast<float>(p0), static_cast<float>(p1), code, stream); }));
}

Call act_backward(PyObject* saved, PyObject* d_out, int act, double p0, double p1, at::Tensor& dx) {
    const at::Tensor *s, *g;
    if (!plain_pair(saved, d_out, &s, &g)) return Call::kGeneral;
    dx = at::empty_like(*s);
    const int64_t n = s->size(-1), m = s->numel() / n;
    void *sp = s->data_ptr(), *gp = g->data_ptr(), *dxp = dx.data_ptr(), *stream = stream_of(*s);
    const int code = type_code(*s);
    return outcome(unlocked([&] { return thn_act_bwd(sp, n, gp, n, dxp, n, m, n, act, static_cast<float>(p0), static_cast<float>(p1), code, stream); }));
}

// The one tensor of a call that was made, None where the general way has to make it.
PyObject* as_result(Call call, const at::Tensor& t) {
    if (call == Call::kGeneral) Py_RETURN_NONE;
    return call == Call::kMade ? THPVariable_Wrap(t) : nullptr;
}

// softmax_fwd(x, kind) -> out
PyObject* softmax_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 2)) return nullptr;
    long long kind;
    if (!whole(args[1], &kind)) Py_RETURN_NONE;
    at::Tensor out;
    const Call call = softmax_forward(args[0], static_cast<int>(kind), out);
    return as_result(call, out);
    END_HANDLE_TH_ERRORS
}

// softmax_bwd(y, dout, kind) -> dx
PyObject* softmax_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 3)) return nullptr;
    long long kind;
    if (!whole(args[2], &kind)) Py_RETURN_NONE;
    at::Tensor dx;
    const Call call = softmax_backward(args[0], args[1], static_cast<int>(kind), dx);
    return as_result(call, dx);
    END_HANDLE_TH_ERRORS
}

// act_fwd(x, act, param0, param1) -> out
PyObject* act_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 4)) return nullptr;
    long long act;
    double p0, p1;
    if (!whole(args[1], &act) || !number(args[2], &p0) || !number(args[3], &p1)) Py_RETURN_NONE;
    at::Tensor out;
    const Call call = act_forward(args[0], static_cast<int>(act), p0, p1, out);
    return as_result(call, out);
    END_HANDLE_TH_ERRORS
}

// act_bwd(saved, dout, act, param0, param1) -> dx
PyObject* act_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 5)) return nullptr;
    long long act;
    double p0, p1;
    if (!whole(args[2], &act) || !number(args[3], &p0) || !number(args[4], &p1)) Py_RETURN_NONE;
    at::Tensor dx;
    const Call call = act_backward(args[0], args[1], static_cast<int>(act), p0, p1, dx);
    return as_result(call, dx);
    END_HANDLE_TH_ERRORS
}

// The p-norm of the rows of a (B, M, K) tensor; normalize: y as well.
Call pnorm_forward(PyObject* input, double p, double eps, bool normalize, at::Tensor& norms, at::Tensor& y) {
    const at::Tensor* x = plain(input);
    if (x == nullptr || x->dim() != 3) return Call::kGeneral;
    const int64_t B = x->size(0), M = x->size(1), K = x->size(2);
    if (normalize) y = at::empty({B, M, K}, x->options());
    norms = at::empty({B, M}, x->options());
    void *xp = x->data_ptr(), *np = norms.data_ptr(), *yp = normalize ? y.data_ptr() : nullptr, *stream = stream_of(*x);
    const int code = type_code(*x);
    return outcome(unlocked([&] {
        if (normalize) return thn_normalize_fwd(xp, M * K, K, yp, M * K, K, np, B, M, K, static_cast<float>(p), static_cast<float>(eps), code, stream);
        return thn_pnorm_fwd(xp, M * K, K, np, B, M, K, static_cast<float>(p), static_cast<float>(eps), code, stream);
    }));
}

// saved_y: null for the p-norm by itself, whose upstream gradient has one value per row.
Call pnorm_backward(PyObject* saved_x, PyObject* saved_y, PyObject* saved_norms, PyObject* d_out, double p, at::Tensor& dx) {
    const at::Tensor *x = plain(saved_x), *y = saved_y != nullptr ? plain(saved_y) : nullptr, *norms = plain(saved_norms), *g = plain(d_out);
    if (x == nullptr || norms == nullptr || g == nullptr || x->dim() != 3) return Call::kGeneral;
    const int64_t B = x->size(0), M = x->size(1), K = x->size(2);
    if (norms->dim() != 2 || norms->size(0) != B || norms->size(1) != M || norms->scalar_type() != x->scalar_type() || g->scalar_type() != x->scalar_type()) return Call::kGeneral;
    if (saved_y != nullptr && (y == nullptr || y->sizes() != x->sizes() || y->scalar_type() != x->scalar_type())) return Call::kGeneral;
    if (g->sizes() != (saved_y != nullptr ? x->sizes() : norms->sizes())) return Call::kGeneral;
    dx = at::empty({B, M, K}, x->options());
    void *xp = x->data_ptr(), *yp = address(y), *np = norms->data_ptr(), *gp = g->data_ptr(), *dxp = dx.data_ptr(), *stream = stream_of(*x);
    const int code = type_code(*x);
    return outcome(unlocked([&] {
        if (saved_y != nullptr) return thn_normalize_bwd(xp, M * K, K, yp, M * K, K, np, gp, M * K, K, dxp, M * K, K, B, M, K, static_cast<float>(p), code, stream);
        return thn_pnorm_bwd(xp, M * K, K, np, gp, dxp, M * K, K, B, M, K, static_cast<float>(p), code, stream);
    }));
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

// ---- The autograd Functions (TritonHub/_autograd.py) -------------------------------------------------------------------
// A Function keeps its forward and backward in Python for every form of call and stays the node that torch makes of it: its context, saved
// tensors, hooks and attributes are torch's own.  For ordinary tensors the Python frames on the way are left out:
//   apply     goes to torch's C apply directly where no functorch transform is active (which is what Function.apply finds out), or, where no
//             gradient can follow, makes the call without a context;
//   forward, backward   are made here, with the attributes and saved tensors that the Python ones set; any other form is theirs.
// Half of a small training pass is the autograd engine, whose thread usually runs on another core complex: there every object that the
// backward touches is fetched from the other side.  us per forward + backward over float32 2 x 100 x 128, frames -> none (both threads on
// one complex in brackets): LayerNorm 88 -> 73 (48 -> 41), RMSNorm 77 -> 64 (42 -> 37), LayerNorm + GeLU 88 -> 75, softmax 58 -> 48.5 (31 -> 27),
// GeLU 59 -> 48, dropout, whose Function stays in Python, 58.5 -> 51.5, normalize 98 -> 53 (48 -> 28), norm 91 -> 50; without gradients
// LayerNorm 11.8 -> 8.2, softmax 8.1 -> 6.1, normalize 14.3 -> 7.0.
enum Kind : int { kLayerNorm, kRmsNorm, kSoftmax, kAct, kPnorm, kNormalize, kPython };

struct Function {
    Kind kind;
    int code = 0;                            // softmax kind, activation
    bool epilogue = false;                   // norms: an activation code is the last argument
    bool saves_output = false;               // activations
    std::vector<PyObject*> params;           // names under which the context keeps the arguments behind the tensors
    PyObject *owner, *general, *forward, *backward;   // the class, its Function.apply, its forward and backward in Python
    PyObject* apply = nullptr;               // torch's C apply for the class whose forward is native
};

struct Ref {                                 // an owned reference
    PyObject* p;
    explicit Ref(PyObject* o) : p(o) {}
    Ref(const Ref&) = delete;
    ~Ref() { Py_XDECREF(p); }
    explicit operator bool() const { return p != nullptr; }
};

PyObject *n_to_save, *n_saved_tensors, *n_needs_input_grad, *n_eps, *n_act, *n_p, *n_cache_policy;
PyObject* g_norm_launch_dict = nullptr;      // TritonHub.Normalization._launch: its cache policy
PyObject* g_read_context = nullptr;          // TritonHub._autograd.ReadContext

Function* function_of(PyObject* capsule) { return static_cast<Function*>(PyCapsule_GetPointer(capsule, "TritonHub.Function")); }

// _x_policy_flag() of TritonHub/Normalization/_launch.py
int policy_flag(bool backward_follows) {
    PyObject* policy = PyDict_GetItem(g_norm_launch_dict, n_cache_policy);      // borrowed
    if (policy == nullptr || !PyUnicode_Check(policy)) return THN_X_STREAM;
    if (PyUnicode_CompareWithASCIIString(policy, "auto") == 0) return backward_follows ? THN_X_KEEP : THN_X_STREAM;
    return PyUnicode_CompareWithASCIIString(policy, "keep") == 0 ? THN_X_KEEP : THN_X_STREAM;
}

// What the native forward leaves: the output, and the saved tensors in the order of the Python forward.
struct Forward {
    at::Tensor out;
    PyObject* inputs[3] = {nullptr, nullptr, nullptr};       // saved inputs, borrowed
    int n_inputs = 0;
    bool saves_out = false;
    at::Tensor made[2];                                      // saved besides: statistics, norms
    int n_made = 0;
};

bool gelu_code(PyObject* approximate, int* code) {
    if (!PyUnicode_CheckExact(approximate)) return false;
    *code = PyUnicode_CompareWithASCIIString(approximate, "tanh") == 0 ? THN_ACT_GELU_TANH : THN_ACT_GELU;
    return true;
}

// The activation's code and parameters from its arguments, or from the attributes of its context.
bool act_params(const Function& f, PyObject* const* params, int* code, double* p0, double* p1) {
    *code = f.code;
    *p0 = *p1 = 0.0;
    if (f.code == THN_ACT_GELU && f.params.size() == 1) return gelu_code(params[0], code);
    if (f.params.size() > 0 && !number(params[0], p0)) return false;
    return f.params.size() < 2 || number(params[1], p1);
}

// `any_grad`: some input requires a gradient (as needs_input_grad says, whether gradients are on or not); `saved`: what it leaves will be saved
Call make_forward(const Function& f, PyObject* const* in, Py_ssize_t n, bool any_grad, bool saved, Forward& r) {
    const Py_ssize_t tensors = f.kind == kLayerNorm ? 3 : f.kind == kRmsNorm ? 2 : 1;
    const bool defaults = f.kind == kPnorm || f.kind == kNormalize;              // p and eps may be left out
    const Py_ssize_t want = tensors + static_cast<Py_ssize_t>(f.params.size());
    if (defaults ? n < 1 || n > 3 : n != want) return Call::kGeneral;
    switch (f.kind) {
        case kLayerNorm:
        case kRmsNorm: {
            const bool ln = f.kind == kLayerNorm;
            long long act = -1;
            if (f.epilogue && (!whole(in[tensors + 1], &act) || act < 0)) return Call::kGeneral;
            at::Tensor results[3];
            const Call call = norm_forward(in[0], in[1], ln ? in[2] : Py_None, in[tensors], ln, act, policy_flag(any_grad), saved, results);
            if (call != Call::kMade) return call;
            r.out = std::move(results[0]);
            if (!saved) return call;
            for (Py_ssize_t i = 0; i < tensors; ++i) r.inputs[i] = in[i];
            r.n_inputs = static_cast<int>(tensors);
            if (ln) r.made[r.n_made++] = std::move(results[1]);
            r.made[r.n_made++] = std::move(results[2]);
            return call;
        }
        case kSoftmax:
            r.saves_out = true;
            return softmax_forward(in[0], f.code, r.out);
        case kAct: {
            int code;
            double p0, p1;
            if (!act_params(f, in + 1, &code, &p0, &p1)) return Call::kGeneral;
            r.saves_out = f.saves_output;
            if (!f.saves_output) r.inputs[r.n_inputs++] = in[0];
            return act_forward(in[0], code, p0, p1, r.out);
        }
        case kPnorm:
        case kNormalize: {
            double p = 2.0, eps = 1e-6;
            if ((n > 1 && !number(in[1], &p)) || (n > 2 && !number(in[2], &eps))) return Call::kGeneral;
            at::Tensor norms, y;
            const Call call = pnorm_forward(in[0], p, eps, f.kind == kNormalize, norms, y);
            if (call != Call::kMade) return call;
            r.inputs[r.n_inputs++] = in[0];
            if (f.kind == kNormalize) {
                r.out = std::move(y);
                r.saves_out = true;
                r.made[r.n_made++] = std::move(norms);
            } else {
                r.out = std::move(norms);
                r.saves_out = true;
            }
            return call;
        }
        default: return Call::kGeneral;
    }
}

PyObject* call_python(PyObject* fn, PyObject* const* args, Py_ssize_t n) { return PyObject_Vectorcall(fn, args, static_cast<size_t>(n), nullptr); }

// forward(ctx, *inputs) -> output
PyObject* function_forward(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    const Function& f = *function_of(self);
    if (nargs < 2) return call_python(f.forward, args, nargs);
    PyObject* ctx = args[0];
    bool any_grad = false;
    if (f.kind == kLayerNorm || f.kind == kRmsNorm) {
        const Ref needs(PyObject_GetAttr(ctx, n_needs_input_grad));
        if (!needs) return nullptr;
        if (!PyTuple_Check(needs.p)) return call_python(f.forward, args, nargs);
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(needs.p); ++i) any_grad = any_grad || PyTuple_GET_ITEM(needs.p, i) == Py_True;
    }
    Forward r;
    const Call call = make_forward(f, args + 1, nargs - 1, any_grad, true, r);
    if (call == Call::kGeneral) return call_python(f.forward, args, nargs);
    if (call == Call::kFailed) return nullptr;
    const Ref out(THPVariable_Wrap(r.out));
    const Ref saved(PyTuple_New(r.n_inputs + (r.saves_out ? 1 : 0) + r.n_made));
    if (!out || !saved) return nullptr;
    Py_ssize_t at = 0;
    for (int i = 0; i < r.n_inputs; ++i) PyTuple_SET_ITEM(saved.p, at++, Py_NewRef(r.inputs[i]));
    if (r.saves_out) PyTuple_SET_ITEM(saved.p, at++, Py_NewRef(out.p));
    for (int i = 0; i < r.n_made; ++i) {
        PyObject* t = THPVariable_Wrap(r.made[i]);
        if (t == nullptr) return nullptr;
        PyTuple_SET_ITEM(saved.p, at++, t);
    }
    if (PyObject_SetAttr(ctx, n_to_save, saved.p) < 0) return nullptr;
    PyObject* const* in = args + 1;
    if (f.kind == kLayerNorm || f.kind == kRmsNorm) {
        const int tensors = f.kind == kLayerNorm ? 3 : 2;
        if (PyObject_SetAttr(ctx, n_eps, in[tensors]) < 0 || (f.epilogue && PyObject_SetAttr(ctx, n_act, in[tensors + 1]) < 0)) return nullptr;
    } else if (f.kind == kPnorm || f.kind == kNormalize) {
        const Ref p(nargs > 2 ? Py_NewRef(in[1]) : PyLong_FromLong(2));
        if (!p || PyObject_SetAttr(ctx, n_p, p.p) < 0) return nullptr;
    } else {
        for (size_t i = 0; i < f.params.size(); ++i) {
            if (PyObject_SetAttr(ctx, f.params[i], in[1 + i]) < 0) return nullptr;
        }
    }
    return Py_NewRef(out.p);
    END_HANDLE_TH_ERRORS
}

// A tuple of the gradients, None behind them, as long as the Python backward's.
template <size_t N> PyObject* gradients(const at::Tensor (&tensors)[N], Py_ssize_t count, Py_ssize_t length) {
    PyObject* result = PyTuple_New(length);
    if (result == nullptr) return nullptr;
    for (Py_ssize_t i = 0; i < length; ++i) {
        PyObject* o = i < count && tensors[i].defined() ? THPVariable_Wrap(tensors[i]) : Py_NewRef(Py_None);
        if (o == nullptr) {
            Py_DECREF(result);
            return nullptr;
        }
        PyTuple_SET_ITEM(result, i, o);
    }
    return result;
}

// backward(ctx, d_out) -> gradients.  The Python backward takes every form that is not made here.  The saved tensors are read once (a
// checkpoint's hooks allow no second time): it gets a context that holds them.
PyObject* function_backward(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    const Function& f = *function_of(self);
    if (f.kind == kPython || nargs != 2 || plain(args[1]) == nullptr) return call_python(f.backward, args, nargs);
    PyObject *ctx = args[0], *d_out = args[1];
    const Ref saved(PyObject_GetAttr(ctx, n_saved_tensors));
    if (!saved) return nullptr;
    const auto has = [&](Py_ssize_t n) { return PyTuple_Check(saved.p) && PyTuple_GET_SIZE(saved.p) == n; };
    const auto item = [&](Py_ssize_t i) { return PyTuple_GET_ITEM(saved.p, i); };
    Call call = Call::kGeneral;
    PyObject* result = nullptr;
    if (f.kind == kLayerNorm || f.kind == kRmsNorm) {
        const bool ln = f.kind == kLayerNorm;
        const Ref needs(PyObject_GetAttr(ctx, n_needs_input_grad));
        if (!needs) return nullptr;
        long long act = -1;
        bool fine = has(ln ? 5 : 3) && PyTuple_Check(needs.p) && PyTuple_GET_SIZE(needs.p) >= (ln ? 3 : 2);
        if (f.epilogue) {
            const Ref code(PyObject_GetAttr(ctx, n_act));
            if (!code) return nullptr;
            fine = fine && whole(code.p, &act) && act >= 0;
        }
        if (fine) {
            const auto needed = [&](Py_ssize_t i) { return PyTuple_GET_ITEM(needs.p, i) == Py_True; };
            at::Tensor results[3];
            call = norm_backward(item(0), d_out, item(1), ln ? item(2) : Py_None, ln ? item(3) : Py_None, item(ln ? 4 : 2), ln, act, needed(1), ln && needed(2), results);
            if (call == Call::kMade) result = gradients(results, ln ? 3 : 2, (ln ? 4 : 3) + (f.epilogue ? 1 : 0));
        }
    } else {
        at::Tensor dx[1];
        if (f.kind == kSoftmax && has(1)) {
            call = softmax_backward(item(0), d_out, f.code, dx[0]);
        } else if (f.kind == kAct && has(1)) {
            const Ref first(f.params.size() > 0 ? PyObject_GetAttr(ctx, f.params[0]) : Py_NewRef(Py_None));
            if (!first) return nullptr;
            const Ref second(f.params.size() > 1 ? PyObject_GetAttr(ctx, f.params[1]) : Py_NewRef(Py_None));
            if (!second) return nullptr;
            PyObject* const values[2] = {first.p, second.p};
            int code;
            double p0, p1;
            if (act_params(f, values, &code, &p0, &p1)) call = act_backward(item(0), d_out, code, p0, p1, dx[0]);
        } else if ((f.kind == kPnorm && has(2)) || (f.kind == kNormalize && has(3))) {
            const Ref p(PyObject_GetAttr(ctx, n_p));
            if (!p) return nullptr;
            double value;
            const bool normalize = f.kind == kNormalize;
            if (number(p.p, &value)) call = pnorm_backward(item(0), normalize ? item(1) : nullptr, item(normalize ? 2 : 1), d_out, value, dx[0]);
        }
        if (call == Call::kMade) {
            const Py_ssize_t behind = f.kind == kPnorm || f.kind == kNormalize ? 2 : static_cast<Py_ssize_t>(f.params.size());
            result = behind == 0 ? THPVariable_Wrap(dx[0]) : gradients(dx, 1, 1 + behind);
        }
    }
    if (call != Call::kGeneral) return result;
    PyObject* const parts[2] = {ctx, saved.p};
    const Ref read(call_python(g_read_context, parts, 2));
    if (!read) return nullptr;
    PyObject* const again[2] = {read.p, d_out};
    return call_python(f.backward, again, 2);
    END_HANDLE_TH_ERRORS
}

bool functorch_active() {
    const auto included = c10::impl::tls_local_dispatch_key_set().included_;
    return included.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || included.has(c10::DispatchKey::FuncTorchDynamicLayerBackMode);
}

// apply(cls, *inputs) -> output
PyObject* function_apply(PyObject* self, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    HANDLE_TH_ERRORS
    const Function& f = *function_of(self);
    bool direct = nargs > 1 && args[0] == f.owner && (kwnames == nullptr || PyTuple_GET_SIZE(kwnames) == 0) && !functorch_active();
    bool any_grad = false, tangent = false;
    for (Py_ssize_t i = 1; direct && i < nargs; ++i) {
        if (!THPVariable_Check(args[i])) continue;
        const at::Tensor& t = THPVariable_Unpack(args[i]);
        // a wrapper of a transform that has ended: Function.apply unwraps it
        direct = t.defined() && !t.unsafeGetTensorImpl()->key_set().has(c10::DispatchKey::FuncTorchGradWrapper);
        any_grad = any_grad || (direct && t.requires_grad());
        tangent = tangent || (direct && t._fw_grad(0).defined());
    }
    if (!direct) {
        // (another class: a subclass that inherited this apply)
        if (nargs == 0 || args[0] == f.owner) return PyObject_Vectorcall(f.general, args + (nargs > 0), static_cast<size_t>(nargs > 0 ? nargs - 1 : 0), kwnames);
        const Ref base(PyObject_GetAttrString(f.general, "__func__"));
        return base ? PyObject_Vectorcall(base.p, args, static_cast<size_t>(nargs), kwnames) : nullptr;
    }
    // Nothing follows that a context would be for.  (A tangent is an error of torch's, a tracer and a profiler note the Function.)
    if (f.kind != kPython && !(any_grad && c10::GradMode::is_enabled()) && !tangent && !at::hasCallbacks() && !torch::jit::tracer::isTracing()) {
        Forward r;
        const Call call = make_forward(f, args + 1, nargs - 1, any_grad, false, r);
        if (call != Call::kGeneral) return as_result(call, r.out);
    }
    return PyObject_Vectorcall(f.apply, args + 1, static_cast<size_t>(nargs - 1), nullptr);
    END_HANDLE_TH_ERRORS
}

PyMethodDef forward_def = {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(function_forward)), METH_FASTCALL, nullptr};
PyMethodDef backward_def = {"apply", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(function_backward)), METH_FASTCALL, nullptr};
PyMethodDef apply_def = {"apply", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(function_apply)), METH_FASTCALL | METH_KEYWORDS, nullptr};

// autograd_function(cls, general_apply, kind, code, params, flag) -> (capsule, forward, backward method of the context's class, apply).  A
// Function's parts live as long as the process.
PyObject* autograd_function(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 6)) return nullptr;
    long long kind, code;
    if (!whole(args[2], &kind) || !whole(args[3], &code) || kind < kLayerNorm || kind > kPython || !PyTuple_Check(args[4])) {
        return PyErr_Format(PyExc_TypeError, "autograd_function(cls, general_apply, kind, code, params, flag)");
    }
    auto* f = new Function{};
    f->kind = static_cast<Kind>(kind);
    f->code = static_cast<int>(code);
    f->owner = Py_NewRef(args[0]);
    f->general = Py_NewRef(args[1]);
    f->forward = PyObject_GetAttrString(args[0], "forward");
    f->backward = PyObject_GetAttrString(args[0], "backward");
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[4]); ++i) f->params.push_back(Py_NewRef(PyTuple_GET_ITEM(args[4], i)));
    const bool flag = PyObject_IsTrue(args[5]) == 1;
    f->epilogue = flag && (f->kind == kLayerNorm || f->kind == kRmsNorm);
    f->saves_output = flag && f->kind == kAct;
    const Ref capsule(PyCapsule_New(f, "TritonHub.Function", nullptr));
    if (!capsule || f->forward == nullptr || f->backward == nullptr) return nullptr;
    const Ref forward(PyCFunction_New(&forward_def, capsule.p)), backward(PyCFunction_New(&backward_def, capsule.p)), apply(PyCFunction_New(&apply_def, capsule.p));
    if (!forward || !backward || !apply) return nullptr;
    const Ref method(PyInstanceMethod_New(backward.p));
    return method ? PyTuple_Pack(4, capsule.p, forward.p, method.p, apply.p) : nullptr;
    END_HANDLE_TH_ERRORS
}

// autograd_function_ready(capsule, torch's C apply of the class with the native forward, the module dictionary with the cache policy, ReadContext)
PyObject* autograd_function_ready(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (wrong_count(nargs, 4)) return nullptr;
    Function* f = function_of(args[0]);
    if (f == nullptr) return nullptr;
    if (g_norm_launch_dict == nullptr) g_norm_launch_dict = Py_NewRef(args[2]);
    if (g_read_context == nullptr) g_read_context = Py_NewRef(args[3]);
    f->apply = Py_NewRef(args[1]);
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define THN_METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(NAME)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {THN_METHOD(norm_fwd),    THN_METHOD(norm_bwd), THN_METHOD(softmax_fwd), THN_METHOD(softmax_bwd),
                         THN_METHOD(act_fwd),     THN_METHOD(act_bwd),  THN_METHOD(dropout_fwd), THN_METHOD(dropout_bwd),
                         THN_METHOD(autograd_function), THN_METHOD(autograd_function_ready),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Host side of the operator calls in native code.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    const std::pair<PyObject**, const char*> names[] = {{&n_to_save, "to_save"}, {&n_saved_tensors, "saved_tensors"}, {&n_needs_input_grad, "needs_input_grad"},
                                                        {&n_eps, "eps"}, {&n_act, "act"}, {&n_p, "p"}, {&n_cache_policy, "_cache_policy"}};
    for (const auto& [place, name] : names) {
        if ((*place = PyUnicode_InternFromString(name)) == nullptr) return nullptr;
    }
    return PyModule_Create(&module);
}
