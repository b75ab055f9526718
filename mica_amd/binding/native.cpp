// Launch path of the operators in native code: a CPython module whose functions take the tensors of one plain call,
// check it, allocate the outputs and call the C ABI (include/mica_amd.h) on the current stream.
//
// Why: an eager call through Python checks, torch.empty and ctypes takes 13 - 16 us of host time on the MI355X's
// host, more than most kernels of a request of a few hundred tokens, so such calls were paced by Python.
//
// Contract: a function launches and returns the call's result, or returns None without having launched or allocated
// anything that lives on, or an int, a failed launch's (negative) HIP error.  None means "not the plain form": a
// refused or unusual call (another device than the current one, a tensor subclass, an active dispatch or function
// mode, vmap, a layout that needs a copy, no workspace yet, a miss code).  The caller's Python path then serves or
// refuses it, so what is accepted and how a refusal reads is decided there alone.
#include <Python.h>

#include <mutex>
#include <optional>
#include <unordered_map>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mica_amd.h"

namespace {

using at::Tensor;

constexpr int kMaxDevices = 64;
constexpr long long kI32 = 1ll << 31;

// the C ABI of the library the Python side loaded (bind())
struct Abi {
#define MICA_FN(name) decltype(&mica_##name) name = nullptr;
    MICA_FN(act_quant)
    MICA_FN(mm_i8)
    MICA_FN(rmsnorm_quant)
    MICA_FN(rmsnorm_quant_multi)
    MICA_FN(attention_prefix_workspace_bytes)
    MICA_FN(attention_fwd)
    MICA_FN(attention_fwd_prefix)
    MICA_FN(causal_conv1d)
    MICA_FN(gdn_chunk)
    MICA_FN(gdn_chunk_gate)
    MICA_FN(gdn_workspace_bytes)
    MICA_FN(gdn_gate)
    MICA_FN(gated_rmsnorm_quant)
#undef MICA_FN
} abi;
bool g_bound = false;
bool g_device_ok[kMaxDevices]; // gfx950 devices, named by the Python side

std::mutex g_ws_mu;
struct Workspace {
    void *ptr;
    long long bytes;
};
std::unordered_map<uint64_t, Workspace> g_ws[kMaxDevices]; // stream handle -> the GEMM's split workspace

// what a call's tensors have in common
struct Call {
    int dev = -1;
    hipStream_t stream = nullptr;
};

bool plain(PyObject *o, const Tensor **t) {
    if (!THPVariable_CheckExact(o)) return false;
    const Tensor &v = THPVariable_Unpack(o);
    if (!v.defined() || !v.device().is_cuda() || v.layout() != at::kStrided || !v.unsafeGetTensorImpl()->has_storage() ||
        v.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                                 c10::DispatchKey::FuncTorchBatched,
                                                 c10::DispatchKey::FuncTorchGradWrapper})))
        return false;
    *t = &v;
    return true;
}
// an optional tensor: None leaves *t null
bool plain_opt(PyObject *o, const Tensor **t) {
    *t = nullptr;
    return o == Py_None || plain(o, t);
}

// Whether the call may run here at all, from its first tensor: the current device, a gfx950 one, and no mode that
// watches tensor operations.
bool enter(const Tensor &t, Call &c) {
    c.dev = t.device().index();
    if (!g_bound || c.dev < 0 || c.dev >= kMaxDevices || !g_device_ok[c.dev]) return false;
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() > 0 ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        return false;
    if (c10::hip::current_device() != c.dev) return false;
    c.stream = c10::hip::getCurrentHIPStream(c.dev).stream();
    return true;
}
bool on(const Call &c, const Tensor &t) { return t.device().index() == c.dev; }
bool aligned(const void *p) { return ((uintptr_t)p & 15u) == 0; }
bool aligned(const Tensor &t) { return aligned(t.data_ptr()); }
Tensor make(const Call &c, at::IntArrayRef shape, at::ScalarType dt) {
    return at::empty(shape, at::TensorOptions().dtype(dt).device(at::Device(at::kCUDA, (c10::DeviceIndex)c.dev)));
}
int code(at::ScalarType t) {
    switch (t) {
    case at::kBFloat16: return MICA_BF16;
    case at::kHalf: return MICA_FP16;
    case at::kFloat: return MICA_FP32;
    default: return -1;
    }
}
void *ptr(const Tensor *t) { return t ? t->data_ptr() : nullptr; }
bool vec_f32(const Call &c, const Tensor &t, int64_t n) {
    return t.scalar_type() == at::kFloat && t.is_contiguous() && t.numel() == n && on(c, t);
}

PyObject *none() { Py_RETURN_NONE; }

// the launch itself, without the interpreter lock (a full queue may block it)
template <class F>
int launch(F f) {
    PyThreadState *s = PyEval_SaveThread();
    const int rc = f();
    PyEval_RestoreThread(s);
    return rc;
}
// rc > 0: the Python path repeats the call and reports the miss
PyObject *bad(int rc) { return rc > 0 ? none() : PyLong_FromLong(rc); }
PyObject *wrap(const Tensor &t) { return THPVariable_Wrap(t); }
PyObject *pack(std::initializer_list<PyObject *> v) {
    PyObject *r = PyTuple_New((Py_ssize_t)v.size());
    Py_ssize_t i = 0;
    for (PyObject *o : v) PyTuple_SET_ITEM(r, i++, o);
    return r;
}
PyObject *new_none() { Py_INCREF(Py_None); return Py_None; }

#define MICA_ARGS(n)                                                                                                  \
    if (nargs != (n)) {                                                                                               \
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");                                                \
        return nullptr;                                                                                               \
    }

// act_quant(x, inv_smooth, rounding) -> (q, s)
PyObject *py_act_quant(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    MICA_ARGS(3)
    const Tensor *x, *inv;
    Call c;
    if (!plain(a[0], &x) || !plain_opt(a[1], &inv) || !enter(*x, c)) return none();
    const int dt = code(x->scalar_type());
    if (x->dim() != 2 || dt < 0) return none();
    const long rounding = PyLong_AsLong(a[2]);
    if (rounding != MICA_ROUND_EVEN && rounding != MICA_ROUND_AWAY) return none();
    const int64_t m = x->size(0), k = x->size(1);
    if (x->stride(1) != 1 || (m > 1 && x->stride(0) != k) || m * k >= kI32) return none();
    if (inv && !vec_f32(c, *inv, k)) return none();
    if (!aligned(*x) || (inv && !aligned(*inv))) return none();
    const Tensor q = make(c, {m, k}, at::kChar), s = make(c, {m}, at::kFloat);
    const int rc = launch([&] {
        return abi.act_quant(x->data_ptr(), dt, (int)k, (const float *)ptr(inv), (int8_t *)q.data_ptr(), (int)k,
                             (float *)s.data_ptr(), (int)m, (int)k, (int)rounding, c.stream);
    });
    if (rc) return bad(rc);
    return pack({wrap(q), wrap(s)});
    END_HANDLE_TH_ERRORS
}

// mm_i8(qx, sx, qw, sw, bias, out dtype code, residual, epilogue, workspace wanted) -> out
PyObject *py_mm_i8(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    MICA_ARGS(9)
    const Tensor *qx, *sx, *qw, *sw, *bias, *res;
    Call c;
    if (!plain(a[0], &qx) || !plain(a[1], &sx) || !plain(a[2], &qw) || !plain(a[3], &sw) || !plain_opt(a[4], &bias) ||
        !plain_opt(a[6], &res) || !enter(*qx, c))
        return none();
    const long dt = PyLong_AsLong(a[5]), epi = PyLong_AsLong(a[7]);
    if (dt != MICA_BF16 && dt != MICA_FP16 && dt != MICA_FP32) return none();
    const at::ScalarType odt = dt == MICA_BF16 ? at::kBFloat16 : dt == MICA_FP16 ? at::kHalf : at::kFloat;
    if (qx->dim() != 2 || qw->dim() != 2 || qx->scalar_type() != at::kChar || qw->scalar_type() != at::kChar) return none();
    const int64_t m = qx->size(0), k = qx->size(1), n = qw->size(0);
    if (qw->size(1) != k || qx->stride(1) != 1 || qw->stride(1) != 1 || (m > 1 && qx->stride(0) != k) ||
        (n > 1 && qw->stride(0) != k) || !on(c, *qw) || k % 16 || m * std::max(k, n) >= kI32)
        return none();
    if (!vec_f32(c, *sx, m) || !vec_f32(c, *sw, n) || (bias && !vec_f32(c, *bias, n))) return none();
    if (epi != MICA_EPI_SCALE && epi != MICA_EPI_SILU_MUL) return none();
    const bool silu = epi == MICA_EPI_SILU_MUL;
    if (silu && (n % 128 || dt != MICA_BF16 || bias || res)) return none();
    const int64_t nout = silu ? n / 2 : n;
    if (res && (res->dim() != 2 || res->size(0) != m || res->size(1) != nout || res->scalar_type() != odt ||
                !res->is_contiguous() || !on(c, *res)))
        return none();
    if (!aligned(*qx) || !aligned(*qw) || !aligned(*sx) || !aligned(*sw) || (bias && !aligned(*bias)) ||
        (res && !aligned(*res)))
        return none();
    Workspace ws{nullptr, 0};
    if (PyObject_IsTrue(a[8])) {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        const auto it = g_ws[c.dev].find((uint64_t)(uintptr_t)c.stream);
        if (it == g_ws[c.dev].end()) return none();
        ws = it->second;
    }
    const Tensor out = make(c, {m, nout}, odt);
    const int rc = launch([&] {
        return abi.mm_i8((const int8_t *)qx->data_ptr(), (int)k, (const int8_t *)qw->data_ptr(), (int)k,
                         (const float *)sx->data_ptr(), (const float *)sw->data_ptr(), (const float *)ptr(bias), ptr(res),
                         (int)nout, out.data_ptr(), (int)nout, (int)dt, (int)m, (int)n, (int)k, (int)epi, ws.ptr,
                         ws.bytes, c.stream);
    });
    if (rc) return bad(rc);
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// the row input of the norms: contiguous rows of bf16 / fp16, a [K] weight, an optional residual like x
bool norm_input(const Call &c, const Tensor &x, const Tensor &w, const Tensor *res) {
    if (x.dim() < 1 || !x.is_contiguous() || x.size(-1) < 1) return false;
    if (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf) return false;
    if (code(w.scalar_type()) < 0 || w.numel() != x.size(-1) || !w.is_contiguous() || !on(c, w)) return false;
    if (res && (res->sizes() != x.sizes() || res->scalar_type() != x.scalar_type() || !res->is_contiguous() || !on(c, *res)))
        return false;
    return aligned(x) && aligned(w) && (!res || aligned(*res));
}

// norm(x, weight, eps, residual, offset, inv_smooth, want q, want y, rounding) -> (q, s, y, summed)
PyObject *py_norm(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    MICA_ARGS(9)
    const Tensor *x, *w, *res, *inv;
    Call c;
    if (!plain(a[0], &x) || !plain(a[1], &w) || !plain_opt(a[3], &res) || !plain_opt(a[5], &inv) || !enter(*x, c))
        return none();
    const double eps = PyFloat_AsDouble(a[2]), offset = PyFloat_AsDouble(a[4]);
    const long rounding = PyLong_AsLong(a[8]);
    if (PyErr_Occurred()) return nullptr;
    if (rounding != MICA_ROUND_EVEN && rounding != MICA_ROUND_AWAY) return none();
    if (!norm_input(c, *x, *w, res)) return none();
    const int64_t K = x->size(-1), M = x->numel() / K;
    if (inv && (!vec_f32(c, *inv, K) || !aligned(*inv))) return none();
    const bool wq = PyObject_IsTrue(a[6]), wy = PyObject_IsTrue(a[7]);
    Tensor q, s, y, sum;
    if (wq) q = make(c, {M, K}, at::kChar), s = make(c, {M}, at::kFloat);
    if (wy) y = make(c, x->sizes(), x->scalar_type());
    if (res) sum = make(c, x->sizes(), x->scalar_type());
    const int rc = launch([&] {
        return abi.rmsnorm_quant(x->data_ptr(), code(x->scalar_type()), (int)K, ptr(res), (int)K, w->data_ptr(),
                                 code(w->scalar_type()), (float)offset, (float)eps, (const float *)ptr(inv),
                                 wq ? (int8_t *)q.data_ptr() : nullptr, (int)K, wq ? (float *)s.data_ptr() : nullptr,
                                 wy ? y.data_ptr() : nullptr, (int)K, res ? sum.data_ptr() : nullptr, (int)K, (int)M,
                                 (int)K, (int)rounding, c.stream);
    });
    if (rc) return bad(rc);
    return pack({wq ? wrap(q) : new_none(), wq ? wrap(s) : new_none(), wy ? wrap(y) : new_none(),
                 res ? wrap(sum) : new_none()});
    END_HANDLE_TH_ERRORS
}

// norm_multi(x, weight, eps, inv_smooths, residual, offset, rounding) -> ([(q, s), ...], summed)
PyObject *py_norm_multi(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    MICA_ARGS(7)
    const Tensor *x, *w, *res;
    Call c;
    if (!PyList_Check(a[3]) || !plain(a[0], &x) || !plain(a[1], &w) || !plain_opt(a[4], &res) || !enter(*x, c))
        return none();
    const double eps = PyFloat_AsDouble(a[2]), offset = PyFloat_AsDouble(a[5]);
    const long rounding = PyLong_AsLong(a[6]);
    if (PyErr_Occurred()) return nullptr;
    const int n = (int)PyList_GET_SIZE(a[3]);
    if (n < 1 || n > 4 || (rounding != MICA_ROUND_EVEN && rounding != MICA_ROUND_AWAY) || !norm_input(c, *x, *w, res))
        return none();
    const int64_t K = x->size(-1), M = x->numel() / K;
    Tensor q[4], s[4], sum;
    const float *invs[4];
    int8_t *qp[4];
    float *sp[4];
    int ld[4];
    for (int i = 0; i < n; ++i) {
        const Tensor *inv;
        if (!plain_opt(PyList_GET_ITEM(a[3], i), &inv) || (inv && (!vec_f32(c, *inv, K) || !aligned(*inv)))) return none();
        invs[i] = (const float *)ptr(inv);
    }
    for (int i = 0; i < n; ++i) {
        q[i] = make(c, {M, K}, at::kChar), s[i] = make(c, {M}, at::kFloat);
        qp[i] = (int8_t *)q[i].data_ptr(), sp[i] = (float *)s[i].data_ptr(), ld[i] = (int)K;
    }
    if (res) sum = make(c, x->sizes(), x->scalar_type());
    const int rc = launch([&] {
        return abi.rmsnorm_quant_multi(x->data_ptr(), code(x->scalar_type()), (int)K, ptr(res), (int)K, w->data_ptr(),
                                       code(w->scalar_type()), (float)offset, (float)eps, n, invs, qp, ld, sp, nullptr,
                                       (int)K, res ? sum.data_ptr() : nullptr, (int)K, (int)M, (int)K, (int)rounding,
                                       c.stream);
    });
    if (rc) return bad(rc);
    PyObject *l = PyList_New(n);
    for (int i = 0; i < n; ++i) PyList_SET_ITEM(l, i, pack({wrap(q[i]), wrap(s[i])}));
    return pack({l, res ? wrap(sum) : new_none()});
    END_HANDLE_TH_ERRORS
}

// attention(q, k, v, 'bshd' layout, scale, prefix k, prefix v) -> o: causal, one workgroup per query block
PyObject *py_attention(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    MICA_ARGS(7)
    const Tensor *q, *k, *v, *kp, *vp;
    Call c;
    if (!plain(a[0], &q) || !plain(a[1], &k) || !plain(a[2], &v) || !plain_opt(a[5], &kp) || !plain_opt(a[6], &vp) ||
        !enter(*q, c))
        return none();
    const bool bshd = PyObject_IsTrue(a[3]);
    const double scale = PyFloat_AsDouble(a[4]);
    if (PyErr_Occurred()) return nullptr;
    constexpr int64_t D = 256, kGroup = 4;
    for (const Tensor *t : {q, k, v})
        if (t->dim() != 4 || t->scalar_type() != at::kBFloat16 || t->size(3) != D || t->stride(3) != 1 || !on(c, *t) ||
            !aligned(*t))
            return none();
    const int hd = bshd ? 2 : 1, sd = bshd ? 1 : 2;
    const int64_t B = q->size(0), Sq = q->size(sd), HQ = q->size(hd), HK = k->size(hd);
    int64_t Sk = k->size(sd), P = 0;
    if (k->sizes() != v->sizes() || k->size(0) != B || HQ != kGroup * HK || Sk < Sq) return none();
    if ((kp == nullptr) != (vp == nullptr)) return none();
    if (kp) {
        for (const Tensor *t : {kp, vp})
            if (!bshd || t->dim() != 3 || t->scalar_type() != at::kBFloat16 || t->size(1) != HK || t->size(2) != D ||
                t->stride(2) != 1 || !on(c, *t) || !aligned(*t))
                return none();
        P = kp->size(0);
        if (P == 0 || vp->size(0) != P || P % 32) return none();
        Sk += P;
    }
    const long long nbytes = abi.attention_prefix_workspace_bytes((int)B, (int)Sq, (int)Sk, (int)P, (int)HQ, (int)HK, 1);
    if (nbytes < 0) return none();
    const Tensor o = make(c, {B, Sq, HQ, D}, at::kBFloat16), ws = make(c, {std::max<int64_t>(nbytes, 16)}, at::kByte);
    const long long qs[3] = {q->stride(0), q->stride(hd), q->stride(sd)}, ks[3] = {k->stride(0), k->stride(hd), k->stride(sd)},
                    vs[3] = {v->stride(0), v->stride(hd), v->stride(sd)}, os[3] = {o.stride(0), o.stride(2), o.stride(1)};
    const int rc = launch([&] {
        if (P)
            return abi.attention_fwd_prefix(q->data_ptr(), qs[0], qs[1], qs[2], k->data_ptr(), ks[0], ks[1], ks[2],
                                            v->data_ptr(), vs[0], vs[1], vs[2], kp->data_ptr(), kp->stride(1),
                                            kp->stride(0), vp->data_ptr(), vp->stride(1), vp->stride(0), (int)P,
                                            o.data_ptr(), os[0], os[1], os[2], (int)B, (int)Sq, (int)Sk, (int)HQ, (int)HK,
                                            (int)D, (float)scale, 1, 1, nullptr, ws.data_ptr(), nbytes, c.stream);
        return abi.attention_fwd(q->data_ptr(), qs[0], qs[1], qs[2], k->data_ptr(), ks[0], ks[1], ks[2], v->data_ptr(),
                                 vs[0], vs[1], vs[2], o.data_ptr(), os[0], os[1], os[2], (int)B, (int)Sq, (int)Sk, (int)HQ,
                                 (int)HK, (int)D, (float)scale, 1, ws.data_ptr(), nbytes, c.stream);
    });
    if (rc) return bad(rc);
    return wrap(bshd ? o : o.transpose(1, 2));
    END_HANDLE_TH_ERRORS
}

// conv(x [B, C, T] channel-last, weight, bias, initial_states, want final states, silu, l2norm heads, eps)
// -> (y [B, C, T], final states or None)
PyObject *py_conv(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    MICA_ARGS(8)
    const Tensor *x, *w, *bias, *init;
    Call c;
    if (!plain(a[0], &x) || !plain(a[1], &w) || !plain_opt(a[2], &bias) || !plain_opt(a[3], &init) || !enter(*x, c))
        return none();
    const bool want = PyObject_IsTrue(a[4]), act = PyObject_IsTrue(a[5]);
    const long l2 = PyLong_AsLong(a[6]);
    const double eps = PyFloat_AsDouble(a[7]);
    if (PyErr_Occurred()) return nullptr;
    if (x->dim() != 3 || x->scalar_type() != at::kBFloat16 || x->stride(1) != 1 || w->dim() != 2) return none();
    const int64_t B = x->size(0), C = x->size(1), T = x->size(2), W = w->size(1);
    const int wd = code(w->scalar_type());
    if (w->size(0) != C || !w->is_contiguous() || !on(c, *w) || (wd != MICA_BF16 && wd != MICA_FP32)) return none();
    if (bias && (bias->scalar_type() != w->scalar_type() || bias->numel() != C || !bias->is_contiguous() || !on(c, *bias)))
        return none();
    if (init && (init->dim() != 3 || init->size(0) != B || init->size(1) != C || init->size(2) != W - 1 ||
                 init->scalar_type() != at::kBFloat16 || !init->is_contiguous() || !on(c, *init)))
        return none();
    if (W < 1 || !aligned(*x)) return none();
    Tensor fin;
    if (want) fin = make(c, {B, C, W - 1}, at::kBFloat16);
    const Tensor y = make(c, {B, T, C}, at::kBFloat16);
    const long long sbx = B > 1 ? x->stride(0) : T * x->stride(2);
    const int rc = launch([&] {
        return abi.causal_conv1d(x->data_ptr(), sbx, (int)x->stride(2), w->data_ptr(), ptr(bias), wd, (int)W, ptr(init),
                                 want ? fin.data_ptr() : nullptr, y.data_ptr(), (long long)(T * C), (int)C, (int)B, (int)T, (int)C,
                                 act ? 1 : 0, (int)l2, (float)eps, c.stream);
    });
    if (rc) return bad(rc);
    return pack({wrap(y.transpose(1, 2)), want ? wrap(fin) : new_none()});
    END_HANDLE_TH_ERRORS
}

// [B, T, H, 128] bf16 rows with contiguous heads
bool heads(const Call &c, const Tensor &t, int64_t B, int64_t T, int64_t H) {
    return t.dim() == 4 && t.size(0) == B && t.size(1) == T && t.size(2) == H && t.size(3) == 128 &&
           t.scalar_type() == at::kBFloat16 && t.stride(3) == 1 && t.stride(2) == 128 && on(c, t) && aligned(t);
}

// rows [M, N] of t over its last axis, when they are evenly spaced
bool rows_of(const Tensor &t, int64_t &M, int64_t &N, int64_t &ld) {
    if (t.dim() != 2 || t.stride(1) != 1) return false;
    M = t.size(0), N = t.size(1), ld = t.stride(0);
    return true;
}

// gdn_chunk(q, k, v, g, beta, scale, initial state, want final state), or with (a, b, A_log, dt_bias) in the place of
// (g, beta) -> (o, final state or None)
PyObject *chunk(PyObject *const *a, Py_ssize_t nargs, bool gate) {
    HANDLE_TH_ERRORS
    MICA_ARGS(gate ? 10 : 8)
    PyObject *const *rest = a + (gate ? 7 : 5);
    const Tensor *q, *k, *v, *g, *beta, *A = nullptr, *dt = nullptr, *h0;
    Call c;
    if (!plain(a[0], &q) || !plain(a[1], &k) || !plain(a[2], &v) || !plain(a[3], &g) || !plain(a[4], &beta) ||
        (gate && (!plain(a[5], &A) || !plain(a[6], &dt))) || !plain_opt(rest[1], &h0) || !enter(*q, c))
        return none();
    const double scale = PyFloat_AsDouble(rest[0]);
    if (PyErr_Occurred()) return nullptr;
    if (q->dim() != 4 || v->dim() != 4) return none();
    const int64_t B = q->size(0), T = q->size(1), HK = q->size(2), HV = v->size(2);
    if (HK < 1 || HV % HK || !heads(c, *q, B, T, HK) || !heads(c, *k, B, T, HK) || !heads(c, *v, B, T, HV)) return none();
    int bd = 0;
    int64_t lda = 0, ldb = 0;
    if (gate) { // g and beta are the rows a and b
        int64_t M, N, M2, N2;
        if (!rows_of(*g, M, N, lda) || !rows_of(*beta, M2, N2, ldb) || M != B * T || M2 != M || N != HV || N2 != HV ||
            g->scalar_type() != at::kBFloat16 || beta->scalar_type() != at::kBFloat16 || !on(c, *g) || !on(c, *beta) ||
            !vec_f32(c, *A, HV) || !vec_f32(c, *dt, HV))
            return none();
    } else {
        if (!vec_f32(c, *g, B * T * HV) || g->dim() != 3 || g->size(0) != B || g->size(1) != T) return none();
        bd = code(beta->scalar_type());
        if ((bd != MICA_BF16 && bd != MICA_FP32) || beta->sizes() != g->sizes() || !beta->is_contiguous() || !on(c, *beta))
            return none();
    }
    if (h0 && (!vec_f32(c, *h0, B * HV * 128 * 128) || h0->dim() != 4 || h0->size(0) != B || h0->size(1) != HV ||
               h0->size(2) != 128 || !aligned(*h0)))
        return none();
    const long long nbytes = abi.gdn_workspace_bytes((int)B, (int)T, (int)HV);
    if (nbytes < 0) return none();
    const bool want = PyObject_IsTrue(rest[2]);
    Tensor hT;
    if (want) hT = make(c, {B, HV, 128, 128}, at::kFloat);
    const Tensor o = make(c, {B, T, HV, 128}, at::kBFloat16), ws = make(c, {std::max<int64_t>(nbytes, 16)}, at::kByte);
    auto sb = [&](const Tensor &t) { return (long long)(B > 1 ? t.stride(0) : T * t.stride(1)); };
    float *hp = want ? (float *)hT.data_ptr() : nullptr;
    const int rc = launch([&] {
        if (gate)
            return abi.gdn_chunk_gate(q->data_ptr(), sb(*q), (int)q->stride(1), k->data_ptr(), sb(*k), (int)k->stride(1),
                                      v->data_ptr(), sb(*v), (int)v->stride(1), g->data_ptr(), (int)lda, beta->data_ptr(),
                                      (int)ldb, (const float *)A->data_ptr(), (const float *)dt->data_ptr(),
                                      (const float *)ptr(h0), hp, o.data_ptr(), (float)scale, (int)B, (int)T, (int)HK,
                                      (int)HV, ws.data_ptr(), nbytes, c.stream);
        return abi.gdn_chunk(q->data_ptr(), sb(*q), (int)q->stride(1), k->data_ptr(), sb(*k), (int)k->stride(1), v->data_ptr(),
                             sb(*v), (int)v->stride(1), (const float *)g->data_ptr(), beta->data_ptr(), bd,
                             (const float *)ptr(h0), hp, o.data_ptr(), (float)scale, (int)B, (int)T, (int)HK, (int)HV,
                             ws.data_ptr(), nbytes, c.stream);
    });
    if (rc) return bad(rc);
    return pack({wrap(o), want ? wrap(hT) : new_none()});
    END_HANDLE_TH_ERRORS
}
PyObject *py_gdn_chunk(PyObject *, PyObject *const *a, Py_ssize_t n) { return chunk(a, n, false); }
PyObject *py_gdn_chunk_gate(PyObject *, PyObject *const *a, Py_ssize_t n) { return chunk(a, n, true); }

// gdn_gate(a, b, A_log, dt_bias) -> (g, beta), a and b [M, HV]
PyObject *py_gdn_gate(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    MICA_ARGS(4)
    const Tensor *a, *b, *A, *dt;
    Call c;
    if (!plain(v[0], &a) || !plain(v[1], &b) || !plain(v[2], &A) || !plain(v[3], &dt) || !enter(*a, c)) return none();
    int64_t M, HV, lda, M2, HV2, ldb;
    if (!rows_of(*a, M, HV, lda) || !rows_of(*b, M2, HV2, ldb) || M2 != M || HV2 != HV || !on(c, *b)) return none();
    if (a->scalar_type() != at::kBFloat16 || b->scalar_type() != at::kBFloat16 || !vec_f32(c, *A, HV) || !vec_f32(c, *dt, HV))
        return none();
    const Tensor g = make(c, {M, HV}, at::kFloat), beta = make(c, {M, HV}, at::kBFloat16);
    const int rc = launch([&] {
        return abi.gdn_gate(a->data_ptr(), (int)lda, b->data_ptr(), (int)ldb, (const float *)A->data_ptr(),
                            (const float *)dt->data_ptr(), (float *)g.data_ptr(), beta.data_ptr(), (int)M, (int)HV, c.stream);
    });
    if (rc) return bad(rc);
    return pack({wrap(g), wrap(beta)});
    END_HANDLE_TH_ERRORS
}

// gated_norm(x, z, weight, eps, want y) -> (q, s, y or None), x and z [M, N]
PyObject *py_gated_norm(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    MICA_ARGS(5)
    const Tensor *x, *z, *w;
    Call c;
    if (!plain(a[0], &x) || !plain(a[1], &z) || !plain(a[2], &w) || !enter(*x, c)) return none();
    const double eps = PyFloat_AsDouble(a[3]);
    if (PyErr_Occurred()) return nullptr;
    int64_t M, N, ldx, M2, N2, ldz;
    if (!rows_of(*x, M, N, ldx) || !rows_of(*z, M2, N2, ldz) || M2 != M || N2 != N || !on(c, *z) || !on(c, *w)) return none();
    if (x->scalar_type() != at::kBFloat16 || z->scalar_type() != at::kBFloat16 || w->scalar_type() != at::kBFloat16 ||
        w->numel() != 128 || !w->is_contiguous() || !aligned(*x) || !aligned(*z) || !aligned(*w))
        return none();
    const bool wy = PyObject_IsTrue(a[4]);
    const Tensor q = make(c, {M, N}, at::kChar), s = make(c, {M}, at::kFloat);
    Tensor y;
    if (wy) y = make(c, {M, N}, at::kBFloat16);
    const int rc = launch([&] {
        return abi.gated_rmsnorm_quant(x->data_ptr(), (int)ldx, z->data_ptr(), (int)ldz, w->data_ptr(), (float)eps,
                                       wy ? y.data_ptr() : nullptr, (int)N, (int8_t *)q.data_ptr(), (int)N,
                                       (float *)s.data_ptr(), (int)M, (int)N, c.stream);
    });
    if (rc) return bad(rc);
    return pack({wrap(q), wrap(s), wy ? wrap(y) : new_none()});
    END_HANDLE_TH_ERRORS
}

// bind({name: address}): the loaded library's functions
PyObject *py_bind(PyObject *, PyObject *d) {
    bool all = PyDict_Check(d);
    auto get = [&](const char *name) -> void * {
        PyObject *o = all ? PyDict_GetItemString(d, name) : nullptr;
        if (o == nullptr) { all = false; return nullptr; }
        return PyLong_AsVoidPtr(o);
    };
#define MICA_FN(name) abi.name = (decltype(abi.name))get("mica_" #name);
    MICA_FN(act_quant)
    MICA_FN(mm_i8)
    MICA_FN(rmsnorm_quant)
    MICA_FN(rmsnorm_quant_multi)
    MICA_FN(attention_prefix_workspace_bytes)
    MICA_FN(attention_fwd)
    MICA_FN(attention_fwd_prefix)
    MICA_FN(causal_conv1d)
    MICA_FN(gdn_chunk)
    MICA_FN(gdn_chunk_gate)
    MICA_FN(gdn_workspace_bytes)
    MICA_FN(gdn_gate)
    MICA_FN(gated_rmsnorm_quant)
#undef MICA_FN
    if (PyErr_Occurred()) return nullptr;
    if (!all) {
        PyErr_SetString(PyExc_ValueError, "bind() needs the address of every function");
        return nullptr;
    }
    g_bound = true;
    Py_RETURN_NONE;
}

// device_ok(index): the device is a gfx950 one
PyObject *py_device_ok(PyObject *, PyObject *i) {
    const long d = PyLong_AsLong(i);
    if (PyErr_Occurred()) return nullptr;
    if (d >= 0 && d < kMaxDevices) g_device_ok[d] = true;
    Py_RETURN_NONE;
}

// workspace(device, stream, pointer, bytes): the GEMM's split workspace of a stream, kept by the caller
PyObject *py_workspace(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    MICA_ARGS(4)
    const long d = PyLong_AsLong(a[0]);
    const uint64_t st = PyLong_AsUnsignedLongLong(a[1]);
    void *p = PyLong_AsVoidPtr(a[2]);
    const long long n = PyLong_AsLongLong(a[3]);
    if (PyErr_Occurred()) return nullptr;
    if (d >= 0 && d < kMaxDevices) {
        std::lock_guard<std::mutex> lock(g_ws_mu);
        g_ws[d][st] = Workspace{p, n};
    }
    Py_RETURN_NONE;
}

#define MICA_DEF(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    MICA_DEF("act_quant", py_act_quant),
    MICA_DEF("mm_i8", py_mm_i8),
    MICA_DEF("norm", py_norm),
    MICA_DEF("norm_multi", py_norm_multi),
    MICA_DEF("attention", py_attention),
    MICA_DEF("conv", py_conv),
    MICA_DEF("gdn_chunk", py_gdn_chunk),
    MICA_DEF("gdn_chunk_gate", py_gdn_chunk_gate),
    MICA_DEF("gdn_gate", py_gdn_gate),
    MICA_DEF("gated_norm", py_gated_norm),
    {"bind", py_bind, METH_O, nullptr},
    {"device_ok", py_device_ok, METH_O, nullptr},
    MICA_DEF("workspace", py_workspace),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Launch path of the mica_amd operators", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
