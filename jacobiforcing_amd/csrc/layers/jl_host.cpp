// jl_host.cpp — the host's side of the small launches, called by layer_ops.py in place of its own checks, allocations and foreign calls.  A launch takes the host 3 us here; around it the
// wrappers in Python took 6 more, which bounds steps of a few tokens (one token through Safisun's four layers: 49 launches).
//
// Every function takes the arguments of the wrapper of its name (a batch's fields one by one), looks at everything the wrapper would, allocates the result and launches.  Whatever it does not
// take in full - other types, shapes, layouts or devices, tensor subclasses, a mode that overrides calls, a trace, gradients where the wrapper looks for them, a call that the library refuses - it leaves to the
// wrapper by returning NotImplemented before anything has happened, and the wrapper takes its general way or raises (moe_experts, whose later launches may refuse what the first took, leaves results
// behind that the wrapper forms again).  A launch that failed is raised here.  Nothing is kept between calls but the kernel libraries' addresses (bind).
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <c10/core/GradMode.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <algorithm>
#include <string.h>
#include <vector>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "jf_layers.h"

namespace {

#define JL_HOST_CALLS(X)                                                                                                                              \
    X(jl_linear_small) X(jl_linear_mid_ok) X(jl_linear_mid) X(jl_linear_split_ok) X(jl_linear_split) X(jl_embed_scale) X(jl_add_rmsnorm) X(jl_sandwich_norm) X(jl_output_norm) X(jl_gated_norm) \
    X(jl_gated_act) X(jl_heads_gate) X(jl_latent_prep) X(jl_latent_q_pack) X(jl_token_shift) X(jl_depth_mix_norm) X(jl_short_conv) X(jl_linear_scan) X(jl_latent_heads_run) \
    X(jl_moe_router_blocks) X(jl_moe_router_run) X(jl_linear_mid_gated) X(jl_rms_norm) X(jl_linear_after_ok) X(jl_linear_after_run) X(jl_moe_few_ok) X(jl_moe_few_run) X(jl_moe_gemm) X(jl_moe_gemm_gated) X(jl_qk_norm_append)
#define DECLARE(name) decltype(&name) p_##name;
JL_HOST_CALLS(DECLARE)
#undef DECLARE

using at::Tensor;
constexpr int MAX_ADDENDS = 3;

PyObject *not_taken() { Py_RETURN_NOTIMPLEMENTED; }

// an ordinary GPU tensor: no subclass, no transform's wrapper, memory of its own
bool take(PyObject *o, const Tensor *&t) {
    if (!THPVariable_CheckExact(o)) return false;
    t = &THPVariable_Unpack(o);
    return t->is_cuda() && t->layout() == at::kStrided &&
           !t->key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Python,
                                                      c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Negative, c10::DispatchKey::Conjugate}));
}
bool take_maybe(PyObject *o, const Tensor *&t) {
    t = nullptr;
    return o == Py_None || take(o, t);
}
bool take(PyObject *o, double &v) {
    if (PyFloat_CheckExact(o)) { v = PyFloat_AS_DOUBLE(o); return true; }
    if (!PyLong_CheckExact(o)) return false;
    v = PyLong_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}
bool take(PyObject *o, int64_t &v) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return !overflow;
}
bool take(PyObject *o, int32_t &v) {
    int64_t w;
    if (!take(o, w) || w != (int32_t)w) return false;
    v = (int32_t)w;
    return true;
}
bool take(PyObject *o, bool &v) {
    if (!PyBool_Check(o)) return false;
    v = o == Py_True;
    return true;
}
// a type that the kernels have, or none
bool take_type(PyObject *o, at::ScalarType &t, bool &given) {
    given = o != Py_None;
    if (!given) return true;
    if (!THPDtype_Check(o)) return false;
    t = ((THPDtype *)o)->scalar_type;
    return t == at::kFloat || t == at::kBFloat16;
}

bool known(const Tensor &t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16; }
int code(at::ScalarType t) { return t == at::kFloat ? JL_F32 : JL_BF16; }
int code(const Tensor &t) { return code(t.scalar_type()); }
bool is_float(const Tensor &t) { return t.scalar_type() == at::kFloat; }
bool rows(const Tensor &t, int64_t n, int64_t w) { return t.dim() == 2 && t.size(0) == n && t.size(1) == w; }
bool row_weights(const Tensor *w, int64_t n) { return !w || (is_float(*w) && w->numel() == n && w->is_contiguous()); }      // float [n]
void *at_(const Tensor *t) { return t ? t->data_ptr() : nullptr; }
void *at_(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
bool starts16(const Tensor &t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }
void *stream_of(const Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
// other threads of the program run from here on, while memory is asked for (which may wait for the device) and launches are queued (which may wait for the queue), until back()
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    void back() { if (state) { PyEval_RestoreThread(state); state = nullptr; } }
    ~Unlocked() { back(); }
};
Tensor make(at::IntArrayRef size, at::ScalarType type, const Tensor &like) { return at::empty(size, at::TensorOptions().dtype(type).device(like.device())); }
bool overridden() { return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() || at::tracer::impl::is_dispatch_enabled(); }
PyObject *wrap(const Tensor &t) { return t.defined() ? THPVariable_Wrap(t) : (Py_INCREF(Py_None), Py_None); }

// the addends of a residual update: a list or tuple of (y [N, W] or [N, S, W], float scale [W] or None)
bool take_addends(PyObject *o, int64_t n, int64_t W, jl_addend (&to)[MAX_ADDENDS], int &count, const Tensor **first = nullptr) {
    if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return false;
    const Py_ssize_t k = PySequence_Fast_GET_SIZE(o);
    if (k > MAX_ADDENDS) return false;
    count = (int)k;
    for (int i = 0; i < count; ++i) {
        PyObject *pair = PySequence_Fast_GET_ITEM(o, i);
        const Tensor *y, *scale;
        if (!PyTuple_CheckExact(pair) || PyTuple_GET_SIZE(pair) != 2 || !take(PyTuple_GET_ITEM(pair, 0), y) || !take_maybe(PyTuple_GET_ITEM(pair, 1), scale)) return false;
        const int64_t d = y->dim();
        if ((d != 2 && d != 3) || !known(*y) || !y->is_contiguous() || y->size(0) != n || y->size(d - 1) != W || (d == 3 && y->size(1) < 1) || !row_weights(scale, W)) return false;
        to[i] = {y->data_ptr(), code(*y), d == 2 ? 1 : (int32_t)y->size(1), (const float *)at_(scale)};
        if (first && i == 0) *first = y;
    }
    return true;
}
// angle tables of a rotation by position
bool angles(int32_t rot_dims, const Tensor *cos, const Tensor *sin, int64_t max_pos, int64_t &length) {
    length = 0;
    if (!rot_dims) return true;
    if (!cos || !sin || !is_float(*cos) || !cos->is_contiguous() || cos->dim() != 2 || cos->sizes() != sin->sizes() || cos->size(1) != rot_dims / 2 || max_pos > cos->size(0)) return false;
    length = cos->size(0);
    return true;
}

#define CALL(name, count)                                                                    \
    PyObject *name(PyObject *, PyObject *const *arg, Py_ssize_t n_args) {                   \
        HANDLE_TH_ERRORS                                                                     \
        if (n_args != (count) || overridden()) return not_taken();
#define END_CALL                                                                             \
    END_HANDLE_TH_ERRORS                                                                     \
    }
bool of_sequences(const char *name) { return !strcmp(name, "jl_linear_scan") || !strncmp(name, "jl_moe", 6); }      // in the library of the recurrences and experts
// a call into the library, with `others` unlocked: refused arguments are the wrapper's to report, a failed launch is raised as it is there
decltype(&jl_last_error) p_last_error, p_last_error_seq;
#define RUN(name, ...)                                                                                                                                               \
    do {                                                                                                                                                              \
        const int rc = p_##name(__VA_ARGS__);                                                                                                                        \
        if (rc != JL_OK) {                                                                                                                                            \
            others.back();                                                                                                                                            \
            if (rc == JL_E_INVALID) return not_taken();                                                                                                               \
            return PyErr_Format(PyExc_RuntimeError, "%s: %s", #name, (of_sequences(#name) ? p_last_error_seq : p_last_error)());                                      \
        }                                                                                                                                                             \
    } while (0)
#define NEED(...) do { if (!(__VA_ARGS__)) return not_taken(); } while (0)

// LINEAR_SMALL_ROWS, LINEAR_ONE_TILE, LINEAR_X_BYTES of layer_ops.py, whose rule this is (linear_small)
int64_t small_rows, one_tile, x_bytes;
bool rule_small(int64_t n, int64_t k, int64_t o, int64_t item) {
    const int64_t tile = o <= one_tile || n == 1 ? 16 : o <= 4 * one_tile ? 32 : 64;
    return n > 0 && n <= small_rows && n * k * item * ((o + tile * 256 - 1) / (tile * 256)) <= x_bytes;
}

// where the launch is taken under autocast as well (2), or where that has nothing to see
bool mid_taken(int64_t n, int64_t k, int64_t o) {
    const int ok = p_jl_linear_mid_ok(n, k, o);
    return ok == 2 || (ok && !at::autocast::is_autocast_enabled(at::kCUDA));
}
// x, w, bias, float_out
CALL(linear, 4)
    const Tensor *x, *w, *bias;
    bool as_float = false;
    NEED(take(arg[0], x) && take(arg[1], w) && take_maybe(arg[2], bias) && (arg[3] == Py_None || take(arg[3], as_float)));
    const bool typed = arg[3] == Py_None;
    NEED(x->dim() == 2 && w->dim() == 2 && known(*x) && known(*w));
    const int64_t n = x->size(0), k = x->size(1), o = w->size(0), ld = x->stride(0), size = w->element_size();
    const bool same = w->scalar_type() == x->scalar_type();
    NEED(same || (is_float(*w) && !typed && as_float));
    const bool small = rule_small(n, k, o, size), split = !small && same && is_float(*w) && p_jl_linear_split_ok(n, k, o) && !at::autocast::is_autocast_enabled(at::kCUDA),
               mid = !small && !split && same && !is_float(*x) && mid_taken(n, k, o);
    NEED(small || split || mid);
    NEED(w->size(1) == k && w->is_contiguous() && x->stride(1) == 1 && ld >= k && k > 0 && o > 0 && o <= INT32_MAX && k * size % 16 == 0 && ld * (int64_t)x->element_size() % 16 == 0 && starts16(*x) &&
         starts16(*w) && w->device() == x->device());
    NEED(!bias || (bias->scalar_type() == w->scalar_type() && bias->dim() == 1 && bias->size(0) == o && bias->is_contiguous() && bias->device() == x->device()));
    NEED(!(c10::GradMode::is_enabled() && (x->requires_grad() || w->requires_grad() || (bias && bias->requires_grad()))));
    NEED(!x->_fw_grad(0).defined() && !w->_fw_grad(0).defined() && !(bias && bias->_fw_grad(0).defined()));      // forward-mode tangents
    NEED(small || split || n * ld * size < (int64_t)1 << 32);
    const int mode = typed ? JL_LINEAR_SAME : as_float ? JL_LINEAR_FLOAT : JL_LINEAR_ROUNDED_FLOAT;
    Unlocked others;
    Tensor out = make({n, o}, typed ? x->scalar_type() : at::kFloat, *x);
    void *st = stream_of(*x);
    if (small) RUN(jl_linear_small, x->data_ptr(), code(*x), n, ld, w->data_ptr(), code(*w), (int32_t)k, (int32_t)o, at_(bias), out.data_ptr(), o, mode, st);
    else if (split) RUN(jl_linear_split, (const float *)x->data_ptr(), n, ld, (const float *)w->data_ptr(), (int32_t)k, (int32_t)o, (const float *)at_(bias), (float *)out.data_ptr(), o, st);
    else RUN(jl_linear_mid, x->data_ptr(), code(*x), n, ld, w->data_ptr(), (int32_t)k, (int32_t)o, at_(bias), out.data_ptr(), o, mode, st);
    others.back();
    return wrap(out);
END_CALL

// out += x w^T (linear_add_)
CALL(linear_add, 3)
    const Tensor *out, *x, *w;
    NEED(take(arg[0], out) && take(arg[1], x) && take(arg[2], w));
    NEED(x->dim() == 2 && w->dim() == 2 && out->dim() == 2 && x->scalar_type() == at::kBFloat16 && w->scalar_type() == at::kBFloat16 && out->scalar_type() == at::kBFloat16);
    const int64_t n = x->size(0), k = x->size(1), o = w->size(0), ld = x->stride(0);
    NEED(n > 0 && k > 0 && o > 0 && o <= INT32_MAX && k <= INT32_MAX && p_jl_linear_mid_ok(n, k, o) && !at::autocast::is_autocast_enabled(at::kCUDA));
    NEED(w->size(1) == k && w->is_contiguous() && rows(*out, n, o) && out->is_contiguous() && x->stride(1) == 1 && ld >= k && k % 8 == 0 && ld % 8 == 0 && starts16(*x) && starts16(*w) && starts16(*out) &&
         w->device() == x->device() && out->device() == x->device() && n * ld * 2 < (int64_t)1 << 32 && !out->is_alias_of(*x) && !out->is_alias_of(*w));
    NEED(!(c10::GradMode::is_enabled() && (x->requires_grad() || w->requires_grad() || out->requires_grad())) && (!out->is_inference() || c10::InferenceMode::is_enabled()));
    NEED(!x->_fw_grad(0).defined() && !w->_fw_grad(0).defined() && !out->_fw_grad(0).defined());
    Unlocked others;
    RUN(jl_linear_mid, x->data_ptr(), JL_BF16, n, ld, w->data_ptr(), (int32_t)k, (int32_t)o, nullptr, out->data_ptr(), o, JL_LINEAR_ADD, stream_of(*x));
    others.back();
    if (!out->is_inference()) out->unsafeGetTensorImpl()->bump_version();       // a graph that kept out for its backward is to see the change
    Py_RETURN_TRUE;
END_CALL

// x, y, x0, w, eps, out_dtype
CALL(add_rmsnorm, 6)
    const Tensor *x, *y, *x0, *w;
    double eps;
    at::ScalarType type = at::kFloat;
    bool wanted;
    NEED(take(arg[0], x) && take_maybe(arg[1], y) && take_maybe(arg[2], x0) && take_maybe(arg[3], w) && take(arg[4], eps) && take_type(arg[5], type, wanted));
    NEED(x->dim() == 2 && is_float(*x) && x->is_contiguous());
    const int64_t n = x->size(0), W = x->size(1);
    NEED(n > 0 && W > 0);
    NEED(!y || (known(*y) && y->is_contiguous() && (y->dim() == 2 || y->dim() == 3) && y->size(0) == n && y->size(-1) == W && (y->dim() == 2 || y->size(1) > 0)));
    NEED(!x0 || (x0->sizes() == x->sizes() && is_float(*x0) && x0->is_contiguous()));
    NEED(!wanted || !w || (w->scalar_type() == type && w->numel() == W && w->is_contiguous()));
    Unlocked others;
    Tensor out;
    if (wanted) out = make({n, W}, type, *x);
    RUN(jl_add_rmsnorm, (float *)x->data_ptr(), at_(y), y ? code(*y) : 0, !y ? 0 : y->dim() == 2 ? 1 : (int32_t)y->size(1), (const float *)at_(x0), at_(w), (float)eps, at_(out), code(type), n,
                          (int32_t)W, stream_of(*x));
    others.back();
    return wrap(out);
END_CALL

// x_in, y, w_post, eps, w_next, out_dtype, add_row, out, plain
CALL(sandwich_norm, 9)
    const Tensor *x, *y, *w_post, *w_next, *add_row, *into;
    double eps;
    at::ScalarType type = at::kFloat;
    bool wanted, plain;
    NEED(take(arg[0], x) && take_maybe(arg[1], y) && take_maybe(arg[2], w_post) && take(arg[3], eps) && take_maybe(arg[4], w_next) && take_type(arg[5], type, wanted) && take_maybe(arg[6], add_row) &&
         take_maybe(arg[7], into) && take(arg[8], plain));
    NEED(x->dim() == 2 && is_float(*x) && x->is_contiguous());
    const int64_t n = x->size(0), W = x->size(1);
    NEED(n > 0 && W > 0 && (!y || (rows(*y, n, W) && known(*y) && y->is_contiguous() && w_post)) && row_weights(w_post, W) && row_weights(add_row, W) && row_weights(w_next, W));
    NEED(!into || (rows(*into, n, W) && known(*into) && into->stride(1) == 1));
    NEED(!(into || wanted) || plain || w_next);
    Unlocked others;
    Tensor out;
    if (into) out = *into;
    else if (wanted) out = make({n, W}, type, *x);
    RUN(jl_sandwich_norm, (const float *)x->data_ptr(), (float *)x->data_ptr(), at_(y), y ? code(*y) : 0, (const float *)at_(w_post), (const float *)at_(add_row), (float)eps,
                            (const float *)at_(w_next), at_(out), out.defined() ? code(out) : 0, out.defined() ? out.stride(0) : 0, plain, n, (int32_t)W, stream_of(*x));
    others.back();
    if (into) { Py_INCREF(arg[7]); return arg[7]; }
    return wrap(out);
END_CALL

// x, w, kind, limit, alpha, shift: the unit of a product whose columns are its gates and its linear branches (linear_gated)
CALL(linear_gated, 6)
    const Tensor *x, *w;
    int32_t kind;
    double limit, alpha, shift;
    NEED(take(arg[0], x) && take(arg[1], w) && take(arg[2], kind) && take(arg[3], limit) && take(arg[4], alpha) && take(arg[5], shift));
    NEED(x->dim() == 2 && w->dim() == 2 && x->scalar_type() == at::kBFloat16 && w->scalar_type() == at::kBFloat16);
    const int64_t n = x->size(0), k = x->size(1), o = w->size(0), ld = x->stride(0);
    NEED(n > 0 && k > 0 && o > 1 && o % 2 == 0 && o <= INT32_MAX && k <= INT32_MAX && !rule_small(n, k, o, 2) && p_jl_linear_mid_ok(n, k, o) && !at::autocast::is_autocast_enabled(at::kCUDA));
    NEED(w->size(1) == k && w->is_contiguous() && x->stride(1) == 1 && ld >= k && k % 8 == 0 && ld % 8 == 0 && starts16(*x) && starts16(*w) && w->device() == x->device() && n * ld * 2 < (int64_t)1 << 32);
    NEED(!(c10::GradMode::is_enabled() && (x->requires_grad() || w->requires_grad())) && !x->_fw_grad(0).defined() && !w->_fw_grad(0).defined());
    Unlocked others;
    Tensor out = make({n, o / 2}, at::kBFloat16, *x);
    RUN(jl_linear_mid_gated, x->data_ptr(), JL_BF16, n, ld, w->data_ptr(), (int32_t)k, (int32_t)(o / 2), kind, (float)limit, (float)alpha, (float)shift, out.data_ptr(), o / 2, stream_of(*x));
    others.back();
    return wrap(out);
END_CALL

// x, w, eps
CALL(rms_norm, 3)
    const Tensor *x, *w;
    double eps;
    NEED(take(arg[0], x) && take(arg[1], w) && take(arg[2], eps));
    NEED(x->dim() >= 1 && known(*x) && x->is_contiguous() && w->dim() == 1 && w->scalar_type() == x->scalar_type() && w->is_contiguous() && w->size(0) == x->size(-1) && w->device() == x->device());
    const int64_t W = w->size(0), vec = 16 / x->element_size();
    NEED(W > 0 && W <= 512 * vec && W % vec == 0 && starts16(*x) && starts16(*w) && x->numel() > 0 && !at::autocast::is_autocast_enabled(at::kCUDA) && !(c10::GradMode::is_enabled() && (x->requires_grad() || w->requires_grad())) &&
         !x->_fw_grad(0).defined() && !w->_fw_grad(0).defined());
    Unlocked others;
    Tensor out = at::empty(x->sizes(), x->options());
    RUN(jl_rms_norm, x->data_ptr(), code(*x), w->data_ptr(), (float)eps, out.data_ptr(), x->numel() / W, (int32_t)W, stream_of(*x));
    others.back();
    return wrap(out);
END_CALL

// a product whose rows its launch makes itself: w and bias [O, K], [O], and what linear (without a choice of result) would need of rows that are whole
bool after_taken(const Tensor &w, const Tensor *bias, int64_t n, int64_t k, const Tensor &like, jl_linear_after &a) {
    if (w.dim() != 2 || w.scalar_type() != at::kBFloat16 || !w.is_contiguous() || w.size(1) != k || !starts16(w) || w.device() != like.device() || !p_jl_linear_after_ok(n, k, w.size(0))) return false;
    if (bias && (bias->scalar_type() != at::kBFloat16 || bias->dim() != 1 || bias->size(0) != w.size(0) || !bias->is_contiguous() || bias->device() != like.device())) return false;
    if ((c10::GradMode::is_enabled() && (w.requires_grad() || like.requires_grad() || (bias && bias->requires_grad()))) || w._fw_grad(0).defined() || like._fw_grad(0).defined() || (bias && bias->_fw_grad(0).defined())) return false;
    a.w = w.data_ptr();
    a.bias = at_(bias);
    a.N = (int32_t)n; a.K = (int32_t)k; a.O = (int32_t)w.size(0);
    return !at::autocast::is_autocast_enabled(at::kCUDA);
}
// x, y, w_post, eps, w_next, add_row, w, bias: the updated x and the product
CALL(norm_linear, 8)
    const Tensor *x, *y, *w_post, *w_next, *add_row, *w, *bias;
    double eps;
    NEED(take(arg[0], x) && take_maybe(arg[1], y) && take_maybe(arg[2], w_post) && take(arg[3], eps) && take(arg[4], w_next) && take_maybe(arg[5], add_row) && take(arg[6], w) && take_maybe(arg[7], bias));
    NEED(x->dim() == 2 && is_float(*x) && x->is_contiguous() && starts16(*x));
    const int64_t n = x->size(0), W = x->size(1);
    jl_linear_after a = {};
    NEED(n > 0 && W > 0 && (!y || (rows(*y, n, W) && known(*y) && y->is_contiguous() && starts16(*y) && w_post)) && row_weights(w_post, W) && row_weights(add_row, W) && row_weights(w_next, W) &&
         after_taken(*w, bias, n, W, *x, a));
    Unlocked others;
    Tensor to = make({n, W}, at::kFloat, *x), out = make({n, w->size(0)}, at::kBFloat16, *x);
    a.mode = JL_AFTER_NORM;
    a.x = x->data_ptr(); a.y = at_(y); a.y_dtype = y ? code(*y) : 0; a.x_out = (float *)to.data_ptr(); a.w_post = (const float *)at_(w_post); a.add_row = (const float *)at_(add_row);
    a.w_next = (const float *)w_next->data_ptr(); a.eps = (float)eps; a.out = out.data_ptr();
    RUN(jl_linear_after_run, &a, stream_of(*x));
    others.back();
    return Py_BuildValue("(NN)", wrap(to), wrap(out));
END_CALL

// z, g_col, u_col, F, kind, limit, alpha, shift, w, bias
CALL(act_linear, 10)
    const Tensor *z, *w, *bias;
    int32_t g_col, u_col, F, kind;
    double limit, alpha, shift;
    NEED(take(arg[0], z) && take(arg[1], g_col) && take(arg[2], u_col) && take(arg[3], F) && take(arg[4], kind) && take(arg[5], limit) && take(arg[6], alpha) && take(arg[7], shift) && take(arg[8], w) &&
         take_maybe(arg[9], bias));
    if (u_col < 0) u_col = -1;
    NEED(z->dim() == 2 && z->scalar_type() == at::kBFloat16 && z->stride(1) == 1 && g_col >= 0 && F > 0 && (int64_t)g_col + F <= z->size(1) && (int64_t)u_col + F <= z->size(1) && starts16(*z));
    const int64_t n = z->size(0);
    jl_linear_after a = {};
    NEED(after_taken(*w, bias, n, F, *z, a));
    Unlocked others;
    Tensor out = make({n, w->size(0)}, at::kBFloat16, *z);
    a.mode = JL_AFTER_ACT;
    a.x = z->data_ptr(); a.x_ld = z->stride(0); a.g_col = g_col; a.u_col = u_col; a.kind = kind; a.limit = (float)limit; a.alpha = (float)alpha; a.shift = (float)shift; a.out = out.data_ptr();
    RUN(jl_linear_after_run, &a, stream_of(*z));
    others.back();
    return wrap(out);
END_CALL

// raw, gate, w_norm, eps, act, gate_first, scale, w, bias
CALL(gated_norm_linear, 9)
    const Tensor *raw, *gate, *wn, *w, *bias;
    double eps, scale;
    int32_t act;
    bool gate_first;
    NEED(take(arg[0], raw) && take(arg[1], gate) && take(arg[2], wn) && take(arg[3], eps) && take(arg[4], act) && take(arg[5], gate_first) && take(arg[6], scale) && take(arg[7], w) && take_maybe(arg[8], bias));
    NEED(raw->dim() == 2 && is_float(*raw) && raw->is_contiguous() && starts16(*raw));
    const int64_t n = raw->size(0), C = raw->size(1);
    jl_linear_after a = {};
    NEED(n > 0 && C > 0 && rows(*gate, n, C) && gate->scalar_type() == at::kBFloat16 && gate->stride(1) == 1 && row_weights(wn, C) && after_taken(*w, bias, n, C, *raw, a));
    Unlocked others;
    Tensor out = make({n, w->size(0)}, at::kBFloat16, *raw);
    a.mode = JL_AFTER_GATED_NORM;
    a.x = raw->data_ptr(); a.y = gate->data_ptr(); a.y_ld = gate->stride(0); a.w_next = (const float *)wn->data_ptr(); a.eps = (float)eps; a.kind = act; a.gate_first = gate_first; a.scale = (float)scale;
    a.out = out.data_ptr();
    RUN(jl_linear_after_run, &a, stream_of(*raw));
    others.back();
    return wrap(out);
END_CALL

// x, addends, w, eps, kind, mult, w_next, out_dtype, choices
CALL(output_norm, 9)
    const Tensor *x, *w, *w_next, *first = nullptr, *ids = nullptr, *weights = nullptr;
    jl_addend addends[MAX_ADDENDS];
    int count;
    double eps, mult;
    int32_t kind, experts = 0;
    at::ScalarType type = at::kFloat;
    bool wanted;
    NEED(take(arg[0], x) && x->dim() == 2 && is_float(*x) && x->is_contiguous());
    const int64_t n = x->size(0), W = x->size(1);
    NEED(n > 0 && W > 0 && take_addends(arg[1], n, W, addends, count, &first) && take_maybe(arg[2], w) && take(arg[3], eps) && take(arg[4], kind) && take(arg[5], mult) && take_maybe(arg[6], w_next) &&
         take_type(arg[7], type, wanted));
    NEED(row_weights(w, W) && row_weights(w_next, W) && (w || count == 0));
    if (arg[8] != Py_None) {
        NEED(PyTuple_CheckExact(arg[8]) && PyTuple_GET_SIZE(arg[8]) == 3 && take(PyTuple_GET_ITEM(arg[8], 0), ids) && take(PyTuple_GET_ITEM(arg[8], 1), weights) &&
             take(PyTuple_GET_ITEM(arg[8], 2), experts));
        NEED(first && first->dim() == 3 && rows(*ids, n, first->size(1)) && rows(*weights, n, first->size(1)) && ids->scalar_type() == at::kInt && is_float(*weights) && ids->is_contiguous() &&
             weights->is_contiguous());
    }
    Unlocked others;
    Tensor out;
    if (wanted) out = make({n, W}, type, *x);
    RUN(jl_output_norm, (float *)x->data_ptr(), addends, count, (const int32_t *)at_(ids), (const float *)at_(weights), ids ? (int32_t)ids->size(1) : 0, experts, kind, (const float *)at_(w),
                          (float)mult, (float)eps, (const float *)at_(w_next), at_(out), code(type), n, (int32_t)W, stream_of(*x));
    others.back();
    return wrap(out);
END_CALL

// raw, gate, w, eps, act, gate_first, parts, scale, out
CALL(gated_norm, 9)
    const Tensor *raw, *gate, *w, *into;
    double eps, scale;
    int32_t act, parts;
    bool gate_first;
    NEED(take(arg[0], raw) && take(arg[1], gate) && take(arg[2], w) && take(arg[3], eps) && take(arg[4], act) && take(arg[5], gate_first) && take(arg[6], parts) && take(arg[7], scale) &&
         take_maybe(arg[8], into));
    NEED(raw->dim() == 2 && is_float(*raw) && raw->is_contiguous());
    const int64_t n = raw->size(0), C = raw->size(1);
    NEED(n > 0 && C > 0 && rows(*gate, n, C) && known(*gate) && gate->stride(1) == 1 && row_weights(w, C) && parts >= 1 && C % parts == 0);
    NEED(!into || (rows(*into, n, C) && into->scalar_type() == gate->scalar_type() && into->stride(1) == 1));
    Unlocked others;
    Tensor out = into ? *into : make({n, C}, gate->scalar_type(), *raw);
    RUN(jl_gated_norm, (const float *)raw->data_ptr(), gate->data_ptr(), code(*gate), gate->stride(0), (const float *)w->data_ptr(), (float)eps, act, gate_first, (float)scale, out.data_ptr(),
                         out.stride(0), n, (int32_t)C, parts, stream_of(*raw));
    others.back();
    if (into) { Py_INCREF(arg[8]); return arg[8]; }
    return wrap(out);
END_CALL

// z, g_col, u_col, F, kind, limit, alpha, shift, row_gate
CALL(gated_act, 9)
    const Tensor *z, *row_gate;
    int32_t g_col, u_col, F, kind;
    double limit, alpha, shift;
    NEED(take(arg[0], z) && take(arg[1], g_col) && take(arg[2], u_col) && take(arg[3], F) && take(arg[4], kind) && take(arg[5], limit) && take(arg[6], alpha) && take(arg[7], shift) &&
         take_maybe(arg[8], row_gate));
    if (u_col < 0) u_col = -1;
    NEED(z->dim() == 2 && known(*z) && z->stride(1) == 1 && g_col >= 0 && F > 0 && (int64_t)g_col + F <= z->size(1) && (int64_t)u_col + F <= z->size(1));
    const int64_t n = z->size(0);
    NEED(n > 0 && (!row_gate || (row_gate->scalar_type() == z->scalar_type() && row_gate->dim() > 0 && row_gate->numel() == n && row_gate->size(0) == n)));
    Unlocked others;
    Tensor out = make({n, F}, z->scalar_type(), *z);
    RUN(jl_gated_act, z->data_ptr(), code(*z), n, z->stride(0), g_col, u_col, F, kind, (float)limit, (float)alpha, (float)shift, at_(row_gate), row_gate ? row_gate->stride(0) : 0, out.data_ptr(),
                        stream_of(*z));
    others.back();
    return wrap(out);
END_CALL

// ov, gate
CALL(heads_gate, 2)
    const Tensor *ov, *gate;
    NEED(take(arg[0], ov) && take_maybe(arg[1], gate) && ov->dim() == 3 && known(*ov) && ov->is_contiguous());
    const int64_t H = ov->size(0), n = ov->size(1), Dv = ov->size(2);
    NEED(H > 0 && n > 0 && Dv > 0 && (!gate || (rows(*gate, n, H * Dv) && gate->stride(1) == 1 && gate->scalar_type() == ov->scalar_type())));
    Unlocked others;
    Tensor out = make({n, H * Dv}, ov->scalar_type(), *ov);
    RUN(jl_heads_gate, ov->data_ptr(), at_(gate), gate ? gate->stride(0) : 0, code(*ov), n, (int32_t)H, (int32_t)Dv, out.data_ptr(), stream_of(*ov));
    others.back();
    return wrap(out);
END_CALL

// proj, q_col, Rq, kv_col, R, rd, rot_dims, wq, wkv, eps, N, max_pos, pos, kv_slot, cos, sin, pool, pairing
CALL(latent_prep, 18)
    const Tensor *proj, *wq, *wkv, *pos, *kv_slot, *cos, *sin, *pool;
    int32_t q_col, Rq, kv_col, R, rd, rot_dims, pairing;
    int64_t n, max_pos, length;
    double eps;
    NEED(take(arg[0], proj) && take(arg[1], q_col) && take(arg[2], Rq) && take(arg[3], kv_col) && take(arg[4], R) && take(arg[5], rd) && take(arg[6], rot_dims) && take_maybe(arg[7], wq) &&
         take_maybe(arg[8], wkv) && take(arg[9], eps) && take(arg[10], n) && take(arg[11], max_pos) && take(arg[12], pos) && take(arg[13], kv_slot) && take_maybe(arg[14], cos) &&
         take_maybe(arg[15], sin) && take_maybe(arg[16], pool) && take(arg[17], pairing));
    NEED(proj->dim() == 2 && known(*proj) && proj->is_contiguous() && proj->size(0) == n && n > 0 && Rq >= 0 && (Rq > 0 || pool));
    NEED(Rq == 0 || (wq && wq->numel() == Rq && wq->scalar_type() == proj->scalar_type()));
    NEED(!pool || (wkv && wkv->numel() == R && wkv->scalar_type() == proj->scalar_type() && pool->scalar_type() == proj->scalar_type() && pool->is_contiguous() && pool->dim() > 0 &&
                   pool->size(-1) == (int64_t)R + rd));
    if (!pool) R = rd = rot_dims = 0;
    NEED(angles(rot_dims, cos, sin, max_pos, length));
    Unlocked others;
    Tensor cq;
    if (Rq) cq = make({n, Rq}, proj->scalar_type(), *proj);
    RUN(jl_latent_prep, proj->data_ptr(), code(*proj), n, proj->size(1), q_col, Rq, kv_col, R, rd, rot_dims, Rq ? at_(wq) : nullptr, at_(wkv), (float)eps, (const int32_t *)at_(pos),
                          (const float *)at_(cos), (const float *)at_(sin), length, at_(cq), at_(pool), (const int64_t *)at_(kv_slot), pairing, stream_of(*proj));
    others.back();
    return wrap(cq);
END_CALL

// qa, q, H, D, R, rd, rot_dims, N, max_pos, pos, cos, sin, pairing
CALL(latent_q_pack, 13)
    const Tensor *qa, *q, *pos, *cos, *sin;
    int32_t H, D, R, rd, rot_dims, pairing;
    int64_t n, max_pos, length;
    NEED(take(arg[0], qa) && take(arg[1], q) && take(arg[2], H) && take(arg[3], D) && take(arg[4], R) && take(arg[5], rd) && take(arg[6], rot_dims) && take(arg[7], n) && take(arg[8], max_pos) &&
         take(arg[9], pos) && take_maybe(arg[10], cos) && take_maybe(arg[11], sin) && take(arg[12], pairing));
    NEED(n > 0 && rows(*q, n, (int64_t)H * (D + rd)) && known(*q) && q->stride(1) == 1 && qa->is_contiguous() && qa->dim() == 3 && qa->size(0) == H && qa->size(1) == n && qa->size(2) == R &&
         qa->scalar_type() == q->scalar_type() && angles(rot_dims, cos, sin, max_pos, length));
    Unlocked others;
    Tensor out = make({n, (int64_t)H * (R + rd)}, q->scalar_type(), *q);
    RUN(jl_latent_q_pack, qa->data_ptr(), q->data_ptr(), q->stride(0), code(*q), n, H, D, R, rd, rot_dims, (const int32_t *)at_(pos), (const float *)at_(cos), (const float *)at_(sin), length,
                            out.data_ptr(), pairing, stream_of(*q));
    others.back();
    return wrap(out);
END_CALL

// x (heads of x_head columns), w [H, K, O], x_head, rd, gate, rot_dims, N, max_pos, pos, cos, sin, pairing: the products of latent attention's heads, [N, H * (O + rd)]
CALL(latent_heads, 12)
    const Tensor *x, *w, *gate, *pos, *cos, *sin;
    int32_t x_head, rd, rot_dims, pairing;
    int64_t n, max_pos, length;
    NEED(take(arg[0], x) && take(arg[1], w) && take(arg[2], x_head) && take(arg[3], rd) && take_maybe(arg[4], gate) && take(arg[5], rot_dims) && take(arg[6], n) && take(arg[7], max_pos) &&
         take(arg[8], pos) && take_maybe(arg[9], cos) && take_maybe(arg[10], sin) && take(arg[11], pairing));
    NEED(x->dim() == 2 && x->scalar_type() == at::kBFloat16 && x->stride(1) == 1 && x->size(0) == n && n > 0 && w->dim() == 3 && w->scalar_type() == at::kBFloat16 && w->is_contiguous() && rd >= 0);
    const int64_t H = w->size(0), K = w->size(1), O = w->size(2);
    NEED(H > 0 && K > 0 && O > 0 && H * (O + rd) <= INT32_MAX && x_head >= K + rd && x->size(1) == H * x_head && w->device() == x->device());
    NEED(!gate || (rows(*gate, n, H * O) && gate->stride(1) == 1 && gate->scalar_type() == at::kBFloat16 && rd == 0));
    NEED(angles(rot_dims, cos, sin, max_pos, length));
    NEED(!(c10::GradMode::is_enabled() && (x->requires_grad() || w->requires_grad())));
    Unlocked others;
    Tensor out = make({n, H * (O + rd)}, at::kBFloat16, *x);
    jl_latent_heads a = {};
    a.x = x->data_ptr(); a.w = w->data_ptr(); a.out = out.data_ptr(); a.gate = at_(gate); a.gate_ld = gate ? gate->stride(0) : 0;
    a.pos = (const int32_t *)pos->data_ptr(); a.cos_t = (const float *)at_(cos); a.sin_t = (const float *)at_(sin);
    a.N = n; a.x_ld = x->stride(0); a.out_ld = H * (O + rd); a.H = (int32_t)H; a.K = (int32_t)K; a.O = (int32_t)O; a.x_head = x_head; a.out_head = (int32_t)(O + rd); a.rd = rd;
    a.rot_dims = rot_dims; a.pairing = pairing;
    RUN(jl_latent_heads_run, &a, stream_of(*x));
    others.back();
    return wrap(out);
END_CALL

// float [slots, ..] with `per` values per slot and the batch's slots
bool carries(const Tensor *tail, int64_t per, int64_t max_slot) {
    return tail && is_float(*tail) && tail->is_contiguous() && tail->dim() > 0 && tail->numel() == tail->size(0) * per && max_slot < tail->size(0);
}

// h, mu, N, max_slot, row_req, seq, tail, out_dtype
CALL(token_shift, 8)
    const Tensor *h, *mu, *row_req, *seq, *tail;
    int64_t n, max_slot;
    at::ScalarType type = at::kFloat;
    bool wanted;
    NEED(take(arg[0], h) && take(arg[1], mu) && take(arg[2], n) && take(arg[3], max_slot) && take(arg[4], row_req) && take(arg[5], seq) && take(arg[6], tail) && take_type(arg[7], type, wanted) && wanted);
    NEED(h->dim() == 2 && is_float(*h) && h->is_contiguous() && h->size(0) == n && n > 0 && row_weights(mu, h->size(1)) && carries(tail, h->size(1), max_slot));
    Unlocked others;
    Tensor out = make({n, h->size(1)}, type, *h);
    RUN(jl_token_shift, (const float *)h->data_ptr(), (const float *)mu->data_ptr(), (const int32_t *)row_req->data_ptr(), (const int32_t *)seq->data_ptr(), (float *)tail->data_ptr(), n,
                          (int32_t)h->size(1), out.data_ptr(), code(type), stream_of(*h));
    others.back();
    return wrap(out);
END_CALL

// x_in, addends, mult, streams, depth, mix, x_out, w, eps, out_dtype, want_float, shift (None, or (mu, tail, seq, max_slot) of a batch with one row per request): out, or (out, float) and the shift's
CALL(depth_mix_norm, 12)
    const Tensor *x, *streams, *mix, *x_out, *w, *mu = nullptr, *tail = nullptr, *seq = nullptr;
    jl_addend addends[MAX_ADDENDS];
    int count;
    double mult, eps;
    int32_t depth;
    int64_t max_slot = 0;
    at::ScalarType type = at::kFloat;
    bool wanted, want_float;
    NEED(take(arg[0], x) && x->dim() == 2 && is_float(*x) && x->is_contiguous());
    const int64_t n = x->size(0), W = x->size(1);
    NEED(n > 0 && W > 0 && take_addends(arg[1], n, W, addends, count) && take(arg[2], mult) && take_maybe(arg[3], streams) && take(arg[4], depth) && take_maybe(arg[5], mix) && take_maybe(arg[6], x_out) &&
         take_maybe(arg[7], w) && take(arg[8], eps) && take_type(arg[9], type, wanted) && take(arg[10], want_float));
    const bool written = depth >= 0 || count > 0;
    NEED(!written || (x_out && is_float(*x_out) && x_out->is_contiguous() && x_out->sizes() == x->sizes()));
    NEED(depth < 0 || (streams && is_float(*streams) && streams->is_contiguous() && streams->dim() == 3 && streams->size(1) == n && streams->size(2) == W && depth < streams->size(0) &&
                       (!mix || (is_float(*mix) && mix->is_contiguous() && mix->numel() >= (int64_t)depth + 1))));
    NEED(row_weights(w, W));
    if (arg[11] != Py_None)
        NEED(PyTuple_CheckExact(arg[11]) && PyTuple_GET_SIZE(arg[11]) == 4 && take(PyTuple_GET_ITEM(arg[11], 0), mu) && take(PyTuple_GET_ITEM(arg[11], 1), tail) &&
             take(PyTuple_GET_ITEM(arg[11], 2), seq) && take(PyTuple_GET_ITEM(arg[11], 3), max_slot) && wanted && row_weights(mu, W) && carries(tail, W, max_slot));
    Unlocked others;
    Tensor out, outf, outs;
    if (wanted) out = make({n, W}, type, *x);
    if (want_float) outf = make({n, W}, at::kFloat, *x);
    if (mu) outs = make({n, W}, type, *x);
    RUN(jl_depth_mix_norm, (const float *)x->data_ptr(), addends, count, (float)mult, depth >= 0 ? (float *)at_(streams) : nullptr, depth >= 0 ? n * W : 0, depth,
                             depth >= 0 ? (const float *)at_(mix) : nullptr, written ? (float *)at_(x_out) : nullptr, (const float *)at_(w), (float)eps, at_(out), code(type), (float *)at_(outf), n,
                             (int32_t)W, (const float *)at_(mu), (const int32_t *)at_(seq), (float *)at_(tail), at_(outs), stream_of(*x));
    others.back();
    if (!want_float && !mu) return wrap(out);
    if (want_float && !mu) return Py_BuildValue("(NN)", wrap(out), wrap(outf));
    if (!want_float) return Py_BuildValue("(NN)", wrap(out), wrap(outs));
    return Py_BuildValue("(NNN)", wrap(out), wrap(outf), wrap(outs));
END_CALL

// x, col, C, w, N, B, max_slot, longest portion behind a start, row_req, seq, tail, act, bias, out_dtype
CALL(short_conv, 14)
    const Tensor *x, *w, *row_req, *seq, *tail, *bias;
    int32_t col, C, B, longest, act;
    int64_t n, max_slot;
    at::ScalarType type = at::kFloat;
    bool wanted;
    NEED(take(arg[0], x) && take(arg[1], col) && take(arg[2], C) && take(arg[3], w) && take(arg[4], n) && take(arg[5], B) && take(arg[6], max_slot) && take(arg[7], longest) && take(arg[8], row_req) &&
         take(arg[9], seq) && take_maybe(arg[10], tail) && take(arg[11], act) && take_maybe(arg[12], bias) && take_type(arg[13], type, wanted) && wanted);
    NEED(x->dim() == 2 && known(*x) && x->is_contiguous() && x->size(0) == n && n > 0 && w->dim() == 2 && w->is_contiguous() && w->size(0) == C && w->scalar_type() == x->scalar_type() && col >= 0 &&
         C > 0 && (int64_t)col + C <= x->size(1) && w->size(1) >= 1 && w->size(1) <= 8);
    const int32_t taps = (int32_t)w->size(1);
    NEED(taps == 1 || (tail && is_float(*tail) && tail->is_contiguous() && tail->dim() == 3 && tail->size(1) == taps - 1 && tail->size(2) == C && max_slot < tail->size(0)));
    NEED((!bias || (bias->scalar_type() == x->scalar_type() && bias->numel() == C && bias->is_contiguous())) && (type == at::kFloat || type == x->scalar_type()));
    Unlocked others;
    Tensor out = make({n, C}, type, *x);
    RUN(jl_short_conv, x->data_ptr(), code(*x), x->size(1), col, w->data_ptr(), at_(bias), (const int32_t *)row_req->data_ptr(), (const int32_t *)seq->data_ptr(), B, longest, (float *)at_(tail), n, C,
                         taps, act, out.data_ptr(), code(type), stream_of(*x));
    others.back();
    return wrap(out);
END_CALL

// a step whose portions are all too short for pieces: src, q_col, k_col, v_col, N, B, max_slot, seq, H, G, D, Dv, state, act, decay, dt, a_log, dt_bias, skip
CALL(linear_scan, 19)
    const Tensor *src, *seq, *state, *decay, *dt, *a_log, *dt_bias, *skip;
    int32_t q_col, k_col, v_col, B, H, G, D, Dv, act;
    int64_t n, max_slot;
    NEED(take(arg[0], src) && take(arg[1], q_col) && take(arg[2], k_col) && take(arg[3], v_col) && take(arg[4], n) && take(arg[5], B) && take(arg[6], max_slot) && take(arg[7], seq) && take(arg[8], H) &&
         take(arg[9], G) && take(arg[10], D) && take(arg[11], Dv) && take(arg[12], state) && take(arg[13], act) && take_maybe(arg[14], decay) && take_maybe(arg[15], dt) && take_maybe(arg[16], a_log) &&
         take_maybe(arg[17], dt_bias) && take_maybe(arg[18], skip));
    NEED(src->dim() == 2 && known(*src) && src->stride(1) == 1 && src->size(0) == n && n > 0 && H > 0 && G > 0 && H % G == 0 && D > 0 && Dv > 0 && q_col >= 0 && k_col >= 0 && v_col >= 0);
    const int64_t ld = src->size(1);
    NEED((q_col > k_col ? q_col : k_col) + (int64_t)G * D <= ld && v_col + (int64_t)H * Dv <= ld);
    NEED(is_float(*state) && state->is_contiguous() && state->dim() == 4 && state->size(1) == H && state->size(2) == D && state->size(3) == Dv && max_slot < state->size(0));
    NEED((decay || (dt && a_log && dt_bias)) && row_weights(decay, H) && row_weights(a_log, H) && row_weights(dt_bias, H) && row_weights(skip, H));
    NEED(decay || (rows(*dt, n, H) && dt->stride(1) == 1 && dt->scalar_type() == src->scalar_type()));
    Unlocked others;
    Tensor out = make({n, (int64_t)H * Dv}, at::kFloat, *src);
    jl_scan_args a = {};
    a.src = src->data_ptr(); a.dt = decay ? nullptr : dt->data_ptr(); a.decay = (const float *)at_(decay); a.A_log = (const float *)at_(a_log); a.dt_bias = (const float *)at_(dt_bias);
    a.skip = (const float *)at_(skip); a.seq = (const int32_t *)seq->data_ptr(); a.state = (float *)state->data_ptr(); a.out = (float *)out.data_ptr();
    a.ld = src->stride(0); a.dt_ld = decay ? 0 : dt->stride(0); a.N = n; a.q_col = q_col; a.k_col = k_col; a.v_col = v_col; a.dtype = code(*src); a.act = act; a.B = B; a.H = H; a.G = G; a.D = D; a.Dv = Dv;
    RUN(jl_linear_scan, &a, stream_of(*src));
    others.back();
    return wrap(out);
END_CALL

// embed, ids, scale, want_copy, out, copy_dtype
CALL(embed_scale, 6)
    const Tensor *embed, *ids, *into;
    double scale;
    bool copy, wanted;
    at::ScalarType type = at::kFloat;
    NEED(take(arg[0], embed) && take(arg[1], ids) && take(arg[2], scale) && take(arg[3], copy) && take_maybe(arg[4], into) && take_type(arg[5], type, wanted) && wanted);
    NEED(embed->dim() == 2 && known(*embed) && embed->is_contiguous() && ids->scalar_type() == at::kLong && ids->is_contiguous());
    const int64_t n = ids->numel(), W = embed->size(1);
    NEED(n > 0 && W > 0 && (!into || (is_float(*into) && into->is_contiguous() && rows(*into, n, W))));
    Unlocked others;
    Tensor x = into ? *into : make({n, W}, at::kFloat, *embed), x0;
    if (copy) x0 = make({n, W}, type, *embed);
    const bool wide = type == at::kFloat;
    RUN(jl_embed_scale, embed->data_ptr(), code(*embed), (const int64_t *)ids->data_ptr(), n, (int32_t)W, (float)scale, (float *)x.data_ptr(), wide ? (float *)at_(x0) : nullptr,
                          wide ? nullptr : at_(x0), stream_of(*embed));
    others.back();
    if (into) { Py_INCREF(arg[4]); return Py_BuildValue("(NN)", arg[4], wrap(x0)); }
    return Py_BuildValue("(NN)", wrap(x), wrap(x0));
END_CALL

// proj, q_col, k_col, v_col, H, G, D, Dv, wq, wk, eps, k_cache, v_cache, kv_slot, rot_dims, pairing, N, max_pos, pos (None without a rotation), cos, sin
CALL(qk_norm_append, 21)
    const Tensor *proj, *wq, *wk, *k, *v, *kv_slot, *pos, *cos, *sin;
    int32_t q_col, k_col, v_col, H, G, D, Dv, rot_dims, pairing;
    int64_t n, max_pos, length;
    double eps;
    NEED(take(arg[0], proj) && take(arg[1], q_col) && take(arg[2], k_col) && take(arg[3], v_col) && take(arg[4], H) && take(arg[5], G) && take(arg[6], D) && take(arg[7], Dv) && take(arg[8], wq) &&
         take(arg[9], wk) && take(arg[10], eps) && take(arg[11], k) && take(arg[12], v) && take(arg[13], kv_slot) && take(arg[14], rot_dims) && take(arg[15], pairing) && take(arg[16], n) &&
         take(arg[17], max_pos) && take_maybe(arg[18], pos) && take_maybe(arg[19], cos) && take_maybe(arg[20], sin));
    const at::ScalarType type = proj->scalar_type();
    NEED(proj->dim() == 2 && known(*proj) && proj->is_contiguous() && proj->size(0) > 0 && kv_slot->scalar_type() == at::kLong && kv_slot->numel() == proj->size(0));
    NEED(wq->numel() == (int64_t)H * D && wk->numel() == (int64_t)G * D && wq->scalar_type() == type && wk->scalar_type() == type);
    NEED(k->scalar_type() == type && v->scalar_type() == type && k->is_contiguous() && v->is_contiguous() && k->dim() > 0 && v->dim() > 0 && k->size(-1) == (int64_t)G * D &&
         v->size(-1) == (int64_t)G * Dv && k->size(0) == v->size(0));
    NEED(rot_dims == 0 || (pos && n == proj->size(0) && rot_dims > 0 && rot_dims % 2 == 0 && rot_dims <= D && angles(rot_dims, cos, sin, max_pos, length)));
    Unlocked others;
    Tensor q = make({proj->size(0), (int64_t)H * D}, type, *proj);
    RUN(jl_qk_norm_append, proj->data_ptr(), code(*proj), proj->size(0), proj->size(1), q_col, k_col, v_col, H, G, D, Dv, wq->data_ptr(), wk->data_ptr(), (float)eps, q.data_ptr(), k->data_ptr(),
        v->data_ptr(), (const int64_t *)kv_slot->data_ptr(), rot_dims, pairing, rot_dims ? (const int32_t *)at_(pos) : nullptr, rot_dims ? (const float *)at_(cos) : nullptr,
        rot_dims ? (const float *)at_(sin) : nullptr, stream_of(*proj));
    others.back();
    return wrap(q);
END_CALL

// h, x (tokens of the router's product, or its float logits when w_router is None), w_router, bias, correction, top, scale, w_up, w_down, kind, renorm_eps, gated (None or (kind, limit, alpha, shift)),
// identity, rows per tile, slices of the product.  The rules (tiles, slices, which launches) are the wrapper's
CALL(moe_experts, 15)
    const Tensor *h, *x, *w_router, *bias, *correction, *w_up, *w_down;
    int32_t top, kind, identity, tm, slices, unit = 0;
    double scale, renorm_eps, limit = 0, alpha = 0, shift = 0;
    NEED(take(arg[0], h) && take(arg[1], x) && take_maybe(arg[2], w_router) && take_maybe(arg[3], bias) && take_maybe(arg[4], correction) && take(arg[5], top) && take(arg[6], scale) && take(arg[7], w_up) &&
         take(arg[8], w_down) && take(arg[9], kind) && take(arg[10], renorm_eps) && take(arg[12], identity) && take(arg[13], tm) && take(arg[14], slices));
    const bool gated = arg[11] != Py_None;
    if (gated)
        NEED(PyTuple_CheckExact(arg[11]) && PyTuple_GET_SIZE(arg[11]) == 4 && take(PyTuple_GET_ITEM(arg[11], 0), unit) && take(PyTuple_GET_ITEM(arg[11], 1), limit) &&
             take(PyTuple_GET_ITEM(arg[11], 2), alpha) && take(PyTuple_GET_ITEM(arg[11], 3), shift));
    NEED(h->dim() == 2 && known(*h) && h->is_contiguous() && w_down->dim() == 3 && w_up->dim() == 3 && identity >= 0);
    const int64_t n = h->size(0), W = h->size(1), E = w_down->size(0), ff = w_down->size(2), Er = E + identity, rows_ = n * top;
    NEED(n > 0 && W > 0 && E > 0 && ff > 0 && top >= 1 && top <= Er && tm > 0 && slices >= 1 && Er <= INT32_MAX && W <= INT32_MAX && 2 * ff <= INT32_MAX && rows_ <= INT32_MAX);
    NEED(w_up->size(0) == E && w_up->size(1) == (gated ? 2 : 1) * ff && w_up->size(2) == W && w_down->size(1) == W && w_up->scalar_type() == h->scalar_type() &&
         w_down->scalar_type() == h->scalar_type() && w_up->is_contiguous() && w_down->is_contiguous());
    NEED(row_weights(correction, Er));
    if (w_router) {
        NEED(x->dim() == 2 && known(*x) && x->size(0) == n && x->stride(1) == 1 && x->device() == h->device() && w_router->dim() == 2 && is_float(*w_router) && w_router->is_contiguous() &&
             w_router->size(0) == Er && w_router->size(1) == x->size(1) && row_weights(bias, Er));
    } else NEED(is_float(*x) && x->is_contiguous() && rows(*x, n, Er) && !bias && slices == 1);
    if (tm == 32 && p_jl_moe_few_ok(code(*h), n, (int32_t)Er, top, (int32_t)W, (int32_t)ff) && starts16(*h) && starts16(*w_up) && starts16(*w_down) &&
        (!w_router || (starts16(*x) && starts16(*w_router) && x->size(1) > 0 && x->size(1) % 4 == 0 && x->stride(0) >= x->size(1) && x->stride(0) * x->element_size() % 16 == 0))) {
        Unlocked others;
        Tensor ids = make({n, top}, at::kInt, *h), weights = make({n, top}, at::kFloat, *h), act = make({rows_, ff}, h->scalar_type(), *h), y = make({n, top, W}, at::kFloat, *h);
        jl_moe_few f = {};
        jl_moe_router &a = f.router;
        a.x = x->data_ptr(); a.w = (const float *)at_(w_router); a.bias = (const float *)at_(bias); a.correction = (const float *)at_(correction);
        a.ids = (int32_t *)ids.data_ptr(); a.weights = (float *)weights.data_ptr();
        a.N = n; a.x_ld = x->stride(0); a.x_dtype = code(*x); a.K = (int32_t)x->size(1); a.E = (int32_t)Er; a.experts = (int32_t)E; a.top = top; a.kind = kind;
        a.scale = (float)scale; a.renorm_eps = (float)renorm_eps;
        f.h = h->data_ptr(); f.w_up = w_up->data_ptr(); f.w_down = w_down->data_ptr(); f.act = act.data_ptr(); f.out = (float *)y.data_ptr();
        f.dtype = code(*h); f.W = (int32_t)W; f.ff = (int32_t)ff; f.gated = gated; f.unit = unit; f.limit = (float)limit; f.alpha = (float)alpha; f.shift = (float)shift;
        RUN(jl_moe_few_run, &f, stream_of(*h));
        others.back();
        if (!identity) return wrap(y);
        return Py_BuildValue("(NNN)", wrap(y), wrap(ids), wrap(weights));
    }
    const int64_t max_tiles = rows_ / tm + E, blocks = p_jl_moe_router_blocks(n), lists = rows_ + E + 2 + 2 * max_tiles + blocks * E;
    Unlocked others;
    Tensor ids = make({n, top}, at::kInt, *h), weights = make({n, top}, at::kFloat, *h), list = make({lists + (slices > 1 ? slices * n * Er : 0)}, at::kInt, *h);
    int32_t *perm = (int32_t *)list.data_ptr(), *offsets = perm + rows_, *tile_expert = offsets + E + 2, *tile_row0 = tile_expert + max_tiles;
    jl_moe_router a = {};
    a.x = x->data_ptr(); a.w = (const float *)at_(w_router); a.bias = (const float *)at_(bias); a.correction = (const float *)at_(correction);
    a.ids = (int32_t *)ids.data_ptr(); a.weights = (float *)weights.data_ptr(); a.perm = perm; a.offsets = offsets; a.tile_expert = tile_expert; a.tile_row0 = tile_row0;
    a.counts = tile_row0 + max_tiles; a.parts = (float *)(perm + lists); a.slices = slices;
    a.N = n; a.x_ld = x->stride(0); a.x_dtype = code(*x); a.K = (int32_t)x->size(1); a.E = (int32_t)Er; a.experts = (int32_t)E; a.top = top; a.kind = kind; a.tile_rows = tm;
    a.max_tiles = (int32_t)max_tiles; a.scale = (float)scale; a.renorm_eps = (float)renorm_eps;
    void *st = stream_of(*h);
    RUN(jl_moe_router_run, &a, st);
    Tensor act = make({rows_, ff}, h->scalar_type(), *h), y = make({n, top, W}, at::kFloat, *h);
    if (gated) RUN(jl_moe_gemm_gated, h->data_ptr(), w_up->data_ptr(), code(*h), (int32_t)W, (int32_t)ff, top, perm, offsets, tile_expert, tile_row0, (int32_t)max_tiles, (int32_t)E, tm, unit,
                   (float)limit, (float)alpha, (float)shift, act.data_ptr(), st);
    else RUN(jl_moe_gemm, h->data_ptr(), w_up->data_ptr(), code(*h), 0, (int32_t)W, (int32_t)ff, top, perm, offsets, tile_expert, tile_row0, (int32_t)max_tiles, (int32_t)E, tm, nullptr,
             act.data_ptr(), st);
    RUN(jl_moe_gemm, act.data_ptr(), w_down->data_ptr(), code(*h), 1, (int32_t)ff, (int32_t)W, top, perm, offsets, tile_expert, tile_row0, (int32_t)max_tiles, (int32_t)E, tm, a.weights, y.data_ptr(),
        st);
    others.back();
    if (!identity) return wrap(y);
    return Py_BuildValue("(NNN)", wrap(y), wrap(ids), wrap(weights));
END_CALL

// Fills the jl_attn_args at an address for operands that the wrapper has checked (its launch is the wrapper's): the address, q, k_cache, v_cache, out, tables, tiles, gate, sink, rel, lut, talk,
// scratch, q_pack, then numbers: scale, softcap, out_scale, page_size, H, G, Gv, D, Dv, window, keep_first, chunk, TQ, splits, out_dtype, gate_heads
CALL(attention_args, 30)
    const Tensor *t[13];
    double real[3];
    int32_t whole[13];
    int64_t address;
    NEED(take(arg[0], address) && address);
    for (int i = 0; i < 13; ++i) NEED(i < 6 ? take(arg[1 + i], t[i]) : take_maybe(arg[1 + i], t[i]));
    for (int i = 0; i < 3; ++i) NEED(take(arg[14 + i], real[i]));
    for (int i = 0; i < 13; ++i) NEED(take(arg[17 + i], whole[i]));
    const Tensor *q = t[0], *k = t[1], *v = t[2], *out = t[3], *tables = t[4], *tiles = t[5], *gate = t[6], *sink = t[7], *rel = t[8], *lut = t[9], *talk = t[10], *scratch = t[11], *pack = t[12];
    NEED(q->dim() == 2 && known(*q) && k->dim() == 2 && v->dim() == 2 && out->dim() == 2 && tables->dim() == 2 && tiles->dim() == 2 && (!gate || gate->dim() == 2) && (!rel || rel->dim() == 2));
    jl_attn_args &a = *(jl_attn_args *)address;
    a = {};
    a.q = q->data_ptr(); a.k_cache = k->data_ptr(); a.v_cache = v->data_ptr(); a.out = out->data_ptr(); a.block_tables = (const int32_t *)tables->data_ptr(); a.tiles = (const int32_t *)tiles->data_ptr();
    a.gate = at_(gate); a.gate_ld = gate ? gate->stride(0) : 0; a.sink = (const float *)at_(sink); a.rel = (const float *)at_(rel); a.lut = (const int32_t *)at_(lut); a.talk = (const float *)at_(talk);
    a.scratch = (float *)at_(scratch); a.q_pack = at_(pack);
    a.lut_len = !rel ? 0 : (int32_t)(lut ? lut->numel() : rel->size(0));
    a.scale = (float)real[0]; a.softcap = (float)real[1]; a.out_scale = (float)real[2];
    a.page_size = whole[0]; a.H = whole[1]; a.G = whole[2]; a.Gv = whole[3]; a.D = whole[4]; a.Dv = whole[5]; a.window = whole[6]; a.keep_first = whole[7]; a.chunk = whole[8]; a.TQ = whole[9];
    a.splits = whole[10]; a.out_dtype = whole[11]; a.gate_heads = whole[12];
    a.bt_stride = tables->size(1); a.n_tiles = (int32_t)tiles->size(0); a.n_rows = q->size(0); a.k_ld = k->stride(0); a.v_ld = v->stride(0); a.out_ld = out->stride(0); a.dtype = code(*q);
    Py_RETURN_NONE;
END_CALL

// ---- a step's tables (RaggedBatch), formed on the host: nothing here touches a device ----------------------------------------------------------------
// a list or tuple of ints within 32 bits
bool take_ints(PyObject *o, std::vector<int64_t> &to) {
    if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return false;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
    to.resize(n);
    for (Py_ssize_t i = 0; i < n; ++i) {
        int32_t v;
        if (!take(PySequence_Fast_GET_ITEM(o, i), v)) return false;
        to[i] = v;
    }
    return true;
}
int64_t fours(int64_t n) { return (n + 3) / 4 * 4; }

// counts, starts, slots, block tables, page size, SCAN_PIECES_FROM -> (the upload as int64, N, columns of the tables, the places of seq, tables, row_req, pos and of a tile per request in it as 32-bit
// words, words of the pieces behind that, largest position, page and slot, longest and shortest portion).  Steps that RaggedBatch.build refuses, and numbers beyond 32 bits, are its own.
CALL(step_tables, 6)
    std::vector<int64_t> counts, starts, slots, held;
    int32_t page, from;
    NEED(take_ints(arg[0], counts) && take_ints(arg[1], starts) && take_ints(arg[2], slots) && (PyList_CheckExact(arg[3]) || PyTuple_CheckExact(arg[3])) && take(arg[4], page) && page > 0 &&
         take(arg[5], from));
    const int64_t B = (int64_t)counts.size(), listed = PySequence_Fast_GET_SIZE(arg[3]);
    NEED(B > 0 && (int64_t)starts.size() == B && (int64_t)slots.size() == B && listed >= B);
    int64_t C = 1, N = 0, longest = 0, least = INT64_MAX, max_pos = 0, max_slot = slots[0];
    held.resize(listed);
    for (int64_t b = 0; b < listed; ++b) {
        PyObject *t = PySequence_Fast_GET_ITEM(arg[3], b);
        NEED(PyList_CheckExact(t) || PyTuple_CheckExact(t));
        held[b] = PySequence_Fast_GET_SIZE(t);
        if (held[b] > C) C = held[b];
        if (b >= B) continue;                                       // tables of more requests count in the width alone
        NEED(counts[b] >= 0 && starts[b] >= 0 && (!counts[b] || (starts[b] + counts[b] + page - 1) / page <= held[b]));
        N += counts[b];
        longest = std::max(longest, counts[b]);
        least = std::min(least, counts[b]);
        max_pos = std::max(max_pos, starts[b] + counts[b]);
        max_slot = std::max(max_slot, slots[b]);
    }
    const int64_t pieced = longest >= from && least > 0 ? 4 * B : 0, sizes[] = {4 * B, B * C, N, N, 4 * B, pieced, pieced};
    int64_t at[8] = {2 * (N + N % 2)};
    for (int i = 0; i < 7; ++i) at[i + 1] = at[i] + fours(sizes[i]);
    NEED(at[7] < INT32_MAX);
    const Tensor up = at::empty({at[7] / 2}, at::TensorOptions().dtype(at::kLong).pinned_memory(false));
    int64_t *pool = up.data_ptr<int64_t>();
    int32_t *words = (int32_t *)pool, *seq = words + at[0], *tables = words + at[1], *req = words + at[2], *pos = words + at[3], *whole = words + at[4], max_page = INT32_MIN;
    memset(words, 0, (size_t)at[7] * 4);
    for (int64_t b = 0, row = 0; b < B; ++b) {
        PyObject *t = PySequence_Fast_GET_ITEM(arg[3], b);
        int32_t *pages = tables + b * C;
        for (int64_t i = 0; i < held[b]; ++i) {
            NEED(take(PySequence_Fast_GET_ITEM(t, i), pages[i]));
            max_page = std::max(max_page, pages[i]);
        }
        for (int64_t i = held[b]; i < C; ++i) pages[i] = -1;
        if (held[b] < C) max_page = std::max(max_page, -1);
        const int32_t c = (int32_t)counts[b], s = (int32_t)starts[b], sl = (int32_t)slots[b], r = (int32_t)row;
        const int32_t s4[] = {r, c, s, sl}, w4[] = {(int32_t)b, s, c, r};
        memcpy(seq + 4 * b, s4, 16);
        memcpy(whole + 4 * b, w4, 16);
        if (pieced) {
            const int32_t piece[] = {r, c, sl, 1}, record[] = {(int32_t)b, 1, s, sl};
            memcpy(words + at[5] + 4 * b, piece, 16);
            memcpy(words + at[6] + 4 * b, record, 16);
        }
        for (int64_t j = s, pg = s / page, in = s % page; j < (int64_t)s + c; ++j, ++row) {
            req[row] = (int32_t)b;
            pos[row] = (int32_t)j;
            pool[row] = (int64_t)pages[pg] * page + in;
            if (++in == page) { in = 0; ++pg; }
        }
    }
    return Py_BuildValue("(NLLLLLLLLLLLLL)", wrap(up), (long long)N, (long long)C, (long long)at[0], (long long)at[1], (long long)at[2], (long long)at[3], (long long)at[4], (long long)pieced,
                         (long long)max_pos, (long long)max_page, (long long)max_slot, (long long)longest, (long long)least);
END_CALL

// the upload, B, N, columns, the places of seq, tables, row_req and pos -> (32-bit words, seq [B, 4], kv_slot [N], tables [B, columns], row_req [N], pos [N])
PyObject *step_views(PyObject *, PyObject *const *arg, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    int64_t B, N, C, at[4];
    if (n_args != 8 || !THPVariable_Check(arg[0]) || !take(arg[1], B) || !take(arg[2], N) || !take(arg[3], C)) return not_taken();
    for (int i = 0; i < 4; ++i) NEED(take(arg[4 + i], at[i]));
    const Tensor &up = THPVariable_Unpack(arg[0]);
    const Tensor words = up.view(at::kInt);
    return Py_BuildValue("(NNNNNN)", wrap(words), wrap(words.as_strided({B, 4}, {4, 1}, at[0])), wrap(up.as_strided({N}, {1}, 0)), wrap(words.as_strided({B, C}, {C, 1}, at[1])),
                         wrap(words.as_strided({N}, {1}, at[2])), wrap(words.as_strided({N}, {1}, at[3])));
END_CALL

// counts, starts, most queries of a tile, whether those with the most positions in front of them come first -> [tiles, 4] int32 {request, first position, count, first row}
CALL(tile_records, 4)
    std::vector<int64_t> counts, starts;
    int32_t tq;
    bool sorted;
    NEED(take_ints(arg[0], counts) && take_ints(arg[1], starts) && counts.size() == starts.size() && take(arg[2], tq) && tq > 0 && take(arg[3], sorted));
    int64_t tiles = 0;
    for (int64_t c : counts) { NEED(c >= 0); tiles += (c + tq - 1) / tq; }
    struct Record { int32_t b, first, count, row; };
    std::vector<Record> records;
    records.reserve(tiles);
    int64_t row = 0;
    for (size_t b = 0; b < counts.size(); ++b) {
        for (int64_t o = 0; o < counts[b]; o += tq)
            records.push_back({(int32_t)b, (int32_t)(starts[b] + o), (int32_t)std::min<int64_t>(tq, counts[b] - o), (int32_t)(row + o)});
        row += counts[b];
    }
    if (sorted) std::stable_sort(records.begin(), records.end(), [](const Record &x, const Record &y) { return x.first > y.first; });
    const Tensor out = at::empty({tiles, 4}, at::TensorOptions().dtype(at::kInt));
    if (tiles) memcpy(out.data_ptr(), records.data(), (size_t)tiles * 16);
    return wrap(out);
END_CALL

// {symbol: address}, LINEAR_SMALL_ROWS, LINEAR_ONE_TILE, LINEAR_X_BYTES
PyObject *bind(PyObject *, PyObject *args) {
    PyObject *symbols;
    long long rows_, tile, bytes;
    if (!PyArg_ParseTuple(args, "O!LLL", &PyDict_Type, &symbols, &rows_, &tile, &bytes)) return nullptr;
    small_rows = rows_; one_tile = tile; x_bytes = bytes;
#define BIND(name)                                                                                                         \
    {                                                                                                                      \
        PyObject *v = PyDict_GetItemString(symbols, #name);                                                                \
        void *p = v ? PyLong_AsVoidPtr(v) : nullptr;                                                                       \
        if (!p) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name); return nullptr; }                         \
        p_##name = (decltype(p_##name))p;                                                                                  \
    }
    JL_HOST_CALLS(BIND)
#undef BIND
    PyObject *e = PyDict_GetItemString(symbols, "jl_last_error"), *q = PyDict_GetItemString(symbols, "jl_last_error of the recurrences");
    if (!e || !q) { PyErr_SetString(PyExc_KeyError, "jl_last_error"); return nullptr; }
    p_last_error = (decltype(p_last_error))PyLong_AsVoidPtr(e);
    p_last_error_seq = (decltype(p_last_error))PyLong_AsVoidPtr(q);
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
}
// n, k, o, bytes of an element, whether x and w are float: which of the package's products linear takes (0: the library's, 1 small, 2 split, 3 mid)
PyObject *linear_rule(PyObject *, PyObject *args) {
    long long n, k, o, item;
    if (!PyArg_ParseTuple(args, "LLLL", &n, &k, &o, &item)) return nullptr;
    return PyLong_FromLong(rule_small(n, k, o, item) ? 1 : item == 4 ? (p_jl_linear_split_ok(n, k, o) ? 2 : 0) : p_jl_linear_mid_ok(n, k, o) ? 3 : 0);
}
PyObject *symbols(PyObject *, PyObject *) {
#define NAME(name) #name,
    static const char *const names[] = {JL_HOST_CALLS(NAME)};
#undef NAME
    PyObject *list = PyList_New(0);
    for (const char *s : names) {
        PyObject *v = list ? PyUnicode_FromString(s) : nullptr;
        if (!v || PyList_Append(list, v)) { Py_XDECREF(v); Py_XDECREF(list); return nullptr; }
        Py_DECREF(v);
    }
    return list;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(linear), FAST(linear_add), FAST(linear_gated), FAST(rms_norm), FAST(norm_linear), FAST(act_linear), FAST(gated_norm_linear), FAST(add_rmsnorm), FAST(sandwich_norm), FAST(output_norm), FAST(gated_norm), FAST(gated_act), FAST(heads_gate), FAST(latent_prep), FAST(latent_q_pack), FAST(latent_heads),
                         FAST(token_shift), FAST(depth_mix_norm), FAST(short_conv), FAST(linear_scan), FAST(embed_scale), FAST(moe_experts), FAST(attention_args), FAST(qk_norm_append), FAST(step_tables), FAST(step_views), FAST(tile_records), {"bind", bind, METH_VARARGS, nullptr},
                         {"linear_rule", linear_rule, METH_VARARGS, nullptr}, {"symbols", symbols, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_jl_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__jl_host() {
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddIntConstant(m, "version", JL_VERSION)) { Py_DECREF(m); return nullptr; }
    return m;
}
