// Native host side of juliavision_amd/kernels.py: an ordinary call goes from torch tensors to the C ABI in here, without
// a Python object per stride, a ctypes conversion per argument or a second planner call.
//
// Every function returns True when it has checked the operands exactly as its Python namesake does, found nothing unusual and
// the library has enqueued the work; False means that nothing was enqueued, and the caller goes on with the Python form,
// which names what is wrong (or carries out what this file does not cover).  Measured on an MI355X host, a 23 x 256 -> 2048
// linear called in a loop: 14.6 us a call through Python checks and three ctypes calls; the kernel itself runs 4.7 us.
//
// `Calls` is a list of C-ABI calls recorded once (by graph.Executor) and issued again with new input addresses.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Device.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <unordered_map>
#include <utility>
#include <vector>
#include "../../include/mi355dnn.h"

namespace {

using at::Tensor;

PyObject *s_dev, *s_own, *s_ws, *s_device, *s_buf, *s_off, *s_scratch;
PyObject *g_workspace_type = nullptr;              // kernels.Workspace: its scratch() is done in here while it need not grow
PyObject *g_ctx_type = nullptr;                    // kernels.Ctx: a subclass may have a stream or a library of its own and goes the long way

// ------------------------------------------------------------------------------------------ operands

const Tensor *tensor(PyObject *o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }
bool is_f16(const Tensor *t) { return t && t->is_cuda() && t->scalar_type() == at::kHalf; }
void *ptr(const Tensor *t) { return t ? t->data_ptr() : nullptr; }

// An operand that may be None: false if it is neither None nor a tensor.
bool optional(PyObject *o, const Tensor *&t) {
    t = nullptr;
    if (o == Py_None) return true;
    t = tensor(o);
    return t != nullptr;
}
bool vec_ok(const Tensor *t, int64_t n, at::ScalarType dtype = at::kHalf) {
    return !t || (t->is_cuda() && t->scalar_type() == dtype && t->numel() == n && t->is_contiguous());
}
bool same_place(const Tensor *r, const Tensor &out) { return !r || (is_f16(r) && r->sizes() == out.sizes() && r->strides() == out.strides()); }
bool dtype_code(const Tensor &t, int &code) {
    if (t.scalar_type() == at::kHalf) code = MI_F16;
    else if (t.scalar_type() == at::kFloat) code = MI_F32;
    else return false;
    return true;
}
// 2-D operand: layout 0 = last axis contiguous, 1 = first axis contiguous
struct Mat { int layout; int64_t ld; };
bool mat2(const Tensor &t, Mat &m) {
    if (t.dim() != 2) return false;
    const auto n = t.sizes();
    const auto s = t.strides();
    if (s[1] == 1 || n[1] == 1) m = {0, n[0] > 1 ? s[0] : std::max<int64_t>(n[1], 1)};
    else if (s[0] == 1) m = {1, n[1] > 1 ? s[1] : std::max<int64_t>(n[0], 1)};
    else return false;
    return true;
}
void strides_elbh(const Tensor &t, int64_t (&s)[4]) {
    const auto st = t.strides();
    s[0] = st[3]; s[1] = st[2]; s[2] = st[1]; s[3] = st[0];
}
bool epi_code(PyObject *o, int &code) {
    if (!PyUnicode_Check(o)) return false;
    static const struct { const char *name; int code; } table[] = {
        {"none", MI_EPI_NONE}, {"gelu", MI_EPI_GELU_ERF}, {"relu", MI_EPI_RELU}, {"gelu_tanh", MI_EPI_GELU_TANH}, {"identity", MI_EPI_NONE}, {"gelu_erf", MI_EPI_GELU_ERF}};
    for (const auto &e : table)
        if (PyUnicode_CompareWithASCIIString(o, e.name) == 0) { code = e.code; return true; }
    return false;
}
bool number(PyObject *o, double &v) {
    v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}
bool pair(PyObject *o, int64_t (&v)[2]) {
    if (PyTuple_CheckExact(o) ? PyTuple_GET_SIZE(o) != 2 : !PyList_CheckExact(o) || PyList_GET_SIZE(o) != 2) return false;
    for (int i = 0; i < 2; i++) {
        PyObject *e = PyTuple_CheckExact(o) ? PyTuple_GET_ITEM(o, i) : PyList_GET_ITEM(o, i);
        if (!PyLong_CheckExact(e)) return false;
        v[i] = PyLong_AsLongLong(e);
        if (v[i] == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    }
    return true;
}

// ------------------------------------------------------------------------------------------ context

// The parts of a kernels.Ctx that a launch needs.  Only a context that plans for the device it was made on (ctx.dev is the
// value it queried; a described device goes the long way) and whose device is the current one is taken.
struct Env {
    void *stream = nullptr;
    PyObject *ws = nullptr;
    ~Env() { Py_XDECREF(ws); }
};
bool env_of(PyObject *ctx, Env &e) {
    if ((PyObject *)Py_TYPE(ctx) != g_ctx_type) return false;
    PyObject *own = PyObject_GetAttr(ctx, s_own), *dev = own ? PyObject_GetAttr(ctx, s_dev) : nullptr;
    const bool mine = own && dev && own == dev && own != Py_None;
    Py_XDECREF(own);
    Py_XDECREF(dev);
    if (!mine) { PyErr_Clear(); return false; }
    PyObject *d = PyObject_GetAttr(ctx, s_device);
    if (!d) { PyErr_Clear(); return false; }
    const int index = THPDevice_Check(d) ? (int)reinterpret_cast<THPDevice *>(d)->device.index() : -2;
    Py_DECREF(d);
    const int cur = (int)c10::hip::current_device();
    if (index != -1 && index != cur) return false;
    e.stream = (void *)c10::hip::getCurrentHIPStream((c10::DeviceIndex)cur).stream();
    e.ws = PyObject_GetAttr(ctx, s_ws);
    if (!e.ws) { PyErr_Clear(); return false; }
    return true;
}
// ws.scratch(need): 256-byte aligned memory of the context's workspace.  False with a Python error set where scratch() raised.
bool scratch(const Env &e, size_t need, void *&p) {
    p = nullptr;
    if (need == 0) return true;
    if ((PyObject *)Py_TYPE(e.ws) == g_workspace_type) {
        PyObject *buf = PyObject_GetAttr(e.ws, s_buf), *off = buf ? PyObject_GetAttr(e.ws, s_off) : nullptr;
        const Tensor *t = buf ? tensor(buf) : nullptr;
        bool done = false;
        if (t && off && PyLong_CheckExact(off)) {
            const uintptr_t base = (uintptr_t)t->data_ptr();
            const int64_t at = PyLong_AsLongLong(off);
            const int64_t start = at + (int64_t)((256 - ((base + (uintptr_t)at) & 255)) & 255);
            if (start + (int64_t)need <= t->numel()) {
                PyObject *next = PyLong_FromLongLong(start + (int64_t)need);
                done = next && PyObject_SetAttr(e.ws, s_off, next) == 0;
                Py_XDECREF(next);
                p = (void *)(base + (uintptr_t)start);
            }
        }
        Py_XDECREF(buf);
        Py_XDECREF(off);
        if (done) return true;
        PyErr_Clear();
    }
    PyObject *n = PyLong_FromSize_t(need), *r = n ? PyObject_CallMethodObjArgs(e.ws, s_scratch, n, nullptr) : nullptr;
    Py_XDECREF(n);
    if (!r) return false;
    p = PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    return !PyErr_Occurred();
}

// A call into the library, with the GIL released as ctypes does: a launch may wait for room in the device's queue.
struct Released {
    PyThreadState *state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
};
template <typename F> int without_gil(F f) {
    Released r;
    return f();
}
#define ANSWER(call) return PyBool_FromLong(without_gil([&] { return call; }) == MI_OK)
#define NO Py_RETURN_FALSE
#define ARITY(n) if (nargs != (n)) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return nullptr; }

// The operands every linear shares: out (T, F), A (K, F) in either layout, B (T, K), bias over features or rows, residual.
struct Linear {
    const Tensor *out, *A, *B, *bias, *res;
    int64_t T, K, F;
    Mat la, lb, lo;
    int layout, bias_mode, epi, out_code;
    size_t need;
};
bool linear_of(Linear &l, PyObject *out, PyObject *A, PyObject *B, PyObject *bias, PyObject *epi, PyObject *res) {
    l.out = tensor(out); l.A = tensor(A); l.B = tensor(B);
    if (!l.out || !is_f16(l.A) || !is_f16(l.B) || !l.out->is_cuda() || !dtype_code(*l.out, l.out_code)) return false;
    if (!mat2(*l.A, l.la) || !mat2(*l.B, l.lb) || !mat2(*l.out, l.lo) || l.lb.layout || l.lo.layout) return false;
    l.K = l.A->size(0); l.F = l.A->size(1); l.T = l.B->size(0);
    if (l.T < 1 || l.K < 1 || l.F < 1 || l.B->size(1) != l.K || l.out->size(0) != l.T || l.out->size(1) != l.F) return false;
    if (!optional(bias, l.bias) || !optional(res, l.res) || !same_place(l.res, *l.out) || !epi_code(epi, l.epi)) return false;
    l.bias_mode = MI_BIAS_NONE;
    if (l.bias) {
        const int64_t n = l.bias->numel();
        if (l.bias->dim() != 1 || (n != l.F && n != l.T) || !vec_ok(l.bias, n)) return false;
        l.bias_mode = n == l.F ? MI_BIAS_COL : MI_BIAS_ROW;
    }
    l.layout = l.la.layout == 0 ? MI_W_KF : MI_W_FK;
    l.need = mi_gemm_f16_workspace(l.T, l.K, l.F, l.layout, 1);
    return true;
}
bool dense(const Tensor &t) { return t.scalar_type() == at::kHalf && t.is_contiguous(); }
bool stats_ok(const Tensor *s, int64_t C, int64_t rows) {
    return s && s->is_cuda() && s->scalar_type() == at::kFloat && s->dim() == 3 && s->size(0) == (C + 31) / 32 && s->size(1) == rows && s->size(2) == 2 && s->is_contiguous();
}

// ------------------------------------------------------------------------------------------ linears

// matmul(ctx, out, A, B, bias, epi, residual)
PyObject *matmul(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(7)
    Linear l;
    Env e;
    void *ws;
    if (!linear_of(l, a[1], a[2], a[3], a[4], a[5], a[6]) || !env_of(a[0], e)) NO;
    if (!scratch(e, l.need, ws)) return nullptr;
    ANSWER(mi_gemm_f16(ptr(l.out), ptr(l.B), ptr(l.A), ptr(l.bias), ptr(l.res), l.T, l.K, l.F, l.lo.ld, l.lb.ld, l.la.ld, l.layout,
                              l.bias_mode, l.epi, l.out_code, ws, l.need, e.stream));
}

// matmul_rowstats(ctx, out, stats, A, B, bias, epi, residual, clamp)
PyObject *matmul_rowstats(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(9)
    Linear l;
    Env e;
    void *ws;
    double clamp = 0.0;
    const Tensor *stats = tensor(a[2]);
    if (!linear_of(l, a[1], a[3], a[4], a[5], a[6], a[7]) || l.T <= 8 || !dense(*l.out) || !stats_ok(stats, l.F, l.T) ||
        (a[8] != Py_None && !number(a[8], clamp)) || !env_of(a[0], e)) NO;
    if (!scratch(e, l.need, ws)) return nullptr;
    ANSWER(mi_gemm_rowstats_f16(ptr(l.out), (float *)ptr(stats), ptr(l.B), ptr(l.A), ptr(l.bias), ptr(l.res), (float)clamp, l.T, l.K, l.F,
                                       l.lb.ld, l.la.ld, l.layout, l.bias_mode, l.epi, ws, l.need, e.stream));
}

// lnfold_matmul(ctx, out, wp, colsum, biasp, planes, B, stats, eps, epi, residual, stats_out, clamp)
PyObject *lnfold_matmul(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(13)
    Linear l;
    Env e;
    void *ws;
    double eps, clamp = 0.0;
    const Tensor *colsum = tensor(a[3]), *biasp = tensor(a[4]), *stats = tensor(a[7]), *stats_out;
    if (!PyLong_CheckExact(a[5]) || !number(a[8], eps) || (a[12] != Py_None && !number(a[12], clamp)) || !optional(a[11], stats_out)) NO;
    const int64_t P = PyLong_AsLongLong(a[5]);
    if (!linear_of(l, a[1], a[2], a[6], Py_None, a[9], a[10]) || P < 1 || l.F % P || !stats_ok(stats, l.K, l.T)) NO;
    if (!colsum || !biasp || !vec_ok(colsum, l.F, at::kFloat) || !vec_ok(biasp, l.F, at::kFloat) || (stats_out && !stats_ok(stats_out, l.F, l.T)) || !env_of(a[0], e)) NO;
    const int64_t Fp = l.F / P, sW = l.layout == MI_W_KF ? Fp : Fp * l.la.ld;
    const size_t need = P == 1 ? l.need : mi_gemm_f16_workspace(l.T, l.K, Fp, l.layout, P);
    if (!scratch(e, need, ws)) return nullptr;
    ANSWER(mi_lnfold_gemm_f16(ptr(l.out), (float *)ptr(stats_out), ptr(l.B), (const float *)ptr(stats), (float)eps, ptr(l.A), (const float *)ptr(colsum),
                                     (const float *)ptr(biasp), ptr(l.res), (float)clamp, l.T, l.K, Fp, l.lo.ld, l.lb.ld, l.la.ld, l.layout, l.epi, l.out_code,
                                     P, Fp, sW, Fp, ws, need, e.stream));
}

// ln_matmul(ctx, out, A, B, gamma, beta, eps, bias, epi, residual): decode-sized rows
PyObject *ln_matmul(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(10)
    Linear l;
    Env e;
    void *ws;
    double eps;
    const Tensor *g, *b;
    if (!linear_of(l, a[1], a[2], a[3], a[7], a[8], a[9]) || l.T > 8 || !optional(a[4], g) || !optional(a[5], b) || !vec_ok(g, l.K) || !vec_ok(b, l.K) ||
        (l.bias && l.bias->numel() != l.F) || !number(a[6], eps) || !env_of(a[0], e)) NO;
    if (!scratch(e, l.need, ws)) return nullptr;
    ANSWER(mi_ln_gemm_f16(ptr(l.out), ptr(l.B), ptr(g), ptr(b), (float)eps, ptr(l.A), ptr(l.bias), ptr(l.res), l.T, l.K, l.F, l.lo.ld, l.lb.ld, l.la.ld,
                                 l.layout, l.bias ? MI_BIAS_COL : MI_BIAS_NONE, l.epi, l.out_code, ws, l.need, e.stream));
}

// ------------------------------------------------------------------------------------------ rows

// layernorm(ctx, out, a, gamma, beta, C, eps), no mean / rstd results
PyObject *layernorm(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(7)
    Env e;
    double eps;
    const Tensor *out = tensor(a[1]), *x = tensor(a[2]), *g, *b;
    if (!is_f16(out) || !is_f16(x) || !out->is_contiguous() || !x->is_contiguous() || out->sizes() != x->sizes() || !PyLong_CheckExact(a[5])) NO;
    const int64_t C = PyLong_AsLongLong(a[5]), n = x->numel();
    if (C < 1 || n % C || !optional(a[3], g) || !optional(a[4], b) || !vec_ok(g, C) || !vec_ok(b, C) || !number(a[6], eps) || !env_of(a[0], e)) NO;
    ANSWER(mi_layernorm_f16(ptr(out), nullptr, nullptr, ptr(x), ptr(g), ptr(b), C, n / C, (float)eps, e.stream));
}

// rowstats(ctx, stats, x)
PyObject *rowstats(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(3)
    Env e;
    const Tensor *s = tensor(a[1]), *x = tensor(a[2]);
    if (!is_f16(x) || x->dim() != 2 || x->stride(1) != 1 || !stats_ok(s, x->size(1), x->size(0)) || !env_of(a[0], e)) NO;
    ANSWER(mi_rowstats_f16((float *)ptr(s), ptr(x), x->stride(0), x->size(1), x->size(0), e.stream));
}

// add(ctx, out, a, b)
PyObject *add(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(4)
    Env e;
    const Tensor *out = tensor(a[1]), *x = tensor(a[2]), *y = tensor(a[3]);
    if (!is_f16(out) || !is_f16(x) || !is_f16(y) || !out->is_contiguous() || !x->is_contiguous() || !y->is_contiguous() || out->sizes() != x->sizes() ||
        out->sizes() != y->sizes() || !env_of(a[0], e)) NO;
    ANSWER(mi_add_f16(ptr(out), ptr(x), ptr(y), x->numel(), e.stream));
}

// ------------------------------------------------------------------------------------------ attention

bool shape_is(const Tensor &t, int64_t a, int64_t b, int64_t c, int64_t d) {
    const auto n = t.sizes();
    return n.size() == 4 && n[0] == a && n[1] == b && n[2] == c && n[3] == d;
}

// sdpa(ctx, q, k, v, bias, scale, out, kv_len)
PyObject *sdpa(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(8)
    Env e;
    void *ws;
    const Tensor *q = tensor(a[1]), *k = tensor(a[2]), *v = tensor(a[3]), *bias, *out = tensor(a[6]), *kv;
    if (!is_f16(q) || !is_f16(k) || !is_f16(v) || q->dim() != 4 || k->dim() != 4 || !optional(a[4], bias) || !optional(a[7], kv)) NO;
    const int64_t B = q->size(0), H = q->size(1), Lq = q->size(2), E = q->size(3), Lk = k->size(2);
    int out_code, bias_code = MI_F16;
    double scale;
    if (B < 1 || H < 1 || Lq < 1 || Lk < 1 || E < 1 || !shape_is(*k, B, H, Lk, E) || !shape_is(*v, B, H, Lk, E)) NO;
    if (!out || !out->is_cuda() || !dtype_code(*out, out_code) || !shape_is(*out, B, H, Lq, E)) NO;
    if (a[5] == Py_None) scale = 1.0 / std::sqrt((double)E);
    else if (!number(a[5], scale)) NO;
    int64_t bs[4] = {0, 0, 0, 0};
    if (bias) {
        if (!bias->is_cuda() || bias->dim() != 4 || !dtype_code(*bias, bias_code)) NO;
        const int64_t full[4] = {Lk, Lq, H, B};
        for (int i = 0; i < 4; i++) {
            const int64_t n = bias->size(3 - i);
            if (n != 1 && n != full[i]) NO;
            bs[i] = n == 1 ? 0 : bias->stride(3 - i);
        }
    }
    if (kv && (kv->scalar_type() != at::kInt || !kv->is_cuda() || kv->numel() != B)) NO;
    if (!env_of(a[0], e)) NO;
    int64_t os[4], qs[4], ks[4], vs[4];
    strides_elbh(*out, os); strides_elbh(*q, qs); strides_elbh(*k, ks); strides_elbh(*v, vs);
    const size_t need = mi_sdpa_f16_workspace(E, Lq, Lk, H, B, bias ? 1 : 0);
    if (!scratch(e, need, ws)) return nullptr;
    ANSWER(mi_sdpa_f16(ptr(out), out_code, out->is_contiguous() ? nullptr : os, ptr(q), qs, ptr(k), ks, ptr(v), vs, ptr(bias), bias_code, bias ? bs : nullptr,
                              (const int32_t *)ptr(kv), E, Lq, Lk, H, B, (float)scale, ws, need, e.stream));
}

// sdpa_append(ctx, q, cache_k, cache_v, k_new, v_new, kv_len, scale, out)
PyObject *sdpa_append(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(9)
    Env e;
    const Tensor *q = tensor(a[1]), *ck = tensor(a[2]), *cv = tensor(a[3]), *kn = tensor(a[4]), *vn = tensor(a[5]), *kv = tensor(a[6]), *out = tensor(a[8]);
    if (!is_f16(q) || !is_f16(ck) || !is_f16(cv) || !is_f16(kn) || !is_f16(vn) || q->dim() != 4 || ck->dim() != 4) NO;
    const int64_t B = q->size(0), H = q->size(1), E = q->size(3), Lk = ck->size(2);
    int out_code;
    double scale;
    if (q->size(2) != 1 || !shape_is(*ck, B, H, Lk, E) || !shape_is(*cv, B, H, Lk, E) || !shape_is(*kn, B, H, 1, E) || !shape_is(*vn, B, H, 1, E) ||
        kn->strides() != vn->strides() || !out || !out->is_cuda() || !dtype_code(*out, out_code) || !shape_is(*out, B, H, 1, E)) NO;
    if (!kv || kv->scalar_type() != at::kInt || !kv->is_cuda() || kv->numel() != B) NO;
    if (a[7] == Py_None) scale = 1.0 / std::sqrt((double)E);
    else if (!number(a[7], scale)) NO;
    if (!env_of(a[0], e)) NO;
    int64_t os[4], qs[4], ks[4], vs[4], ns[4];
    strides_elbh(*out, os); strides_elbh(*q, qs); strides_elbh(*ck, ks); strides_elbh(*cv, vs); strides_elbh(*kn, ns);
    ANSWER(mi_sdpa_append_f16(ptr(out), out_code, out->is_contiguous() ? nullptr : os, ptr(q), qs, ptr(ck), ks, ptr(cv), vs, ptr(kn), ptr(vn), ns,
                                     (const int32_t *)ptr(kv), E, Lk, H, B, (float)scale, e.stream));
}

// ------------------------------------------------------------------------------------------ convolution

bool plain4(const Tensor *t) { return is_f16(t) && t->dim() == 4 && t->is_contiguous(); }
int64_t conv_extent(int64_t n, int64_t k, int64_t s, int64_t p, int64_t d) {
    const int64_t a = n + 2 * p - d * (k - 1) - 1;
    return a < 0 ? 0 : a / s + 1;
}

// convolution(ctx, out, x, w, bias, stride, padding, dilation, groups, act)
PyObject *convolution(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(10)
    Env e;
    void *ws;
    const Tensor *out = tensor(a[1]), *x = tensor(a[2]), *w = tensor(a[3]), *bias;
    int64_t s[2], p[2], d[2];
    int act;
    if (!plain4(out) || !plain4(x) || !plain4(w) || !optional(a[4], bias) || !pair(a[5], s) || !pair(a[6], p) || !pair(a[7], d) || !PyLong_CheckExact(a[8]) ||
        !epi_code(a[9], act)) NO;
    const int64_t groups = PyLong_AsLongLong(a[8]), N = x->size(0), Cin = x->size(1), Hi = x->size(2), Wi = x->size(3), Cout = w->size(0), KH = w->size(2), KW = w->size(3);
    if (groups < 1 || w->size(1) * groups != Cin || s[0] < 1 || s[1] < 1 || x->numel() < 1 || out->numel() < 1 || !vec_ok(bias, Cout)) NO;
    if (!shape_is(*out, N, Cout, conv_extent(Hi, KH, s[1], p[1], d[1]), conv_extent(Wi, KW, s[0], p[0], d[0])) || !env_of(a[0], e)) NO;
    size_t need = 0;
    if (mi_conv2d_f16_kernel(Wi, Hi, Cin, N, KW, KH, Cout, s[0], s[1], p[0], p[1], d[0], d[1], groups, &need) == MI_CONV_KERNEL_NONE) NO;
    if (!scratch(e, need, ws)) return nullptr;
    ANSWER(mi_conv2d_f16(ptr(out), ptr(x), ptr(w), ptr(bias), Wi, Hi, Cin, N, KW, KH, Cout, s[0], s[1], p[0], p[1], d[0], d[1], groups, act, ws, need, e.stream));
}

// convolutiontranspose(ctx, out, x, w, bias, stride, padding, dilation, outpad, groups)
PyObject *convolutiontranspose(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(10)
    Env e;
    const Tensor *out = tensor(a[1]), *x = tensor(a[2]), *w = tensor(a[3]), *bias;
    int64_t s[2], p[2], d[2], o[2];
    if (!plain4(out) || !plain4(x) || !plain4(w) || !optional(a[4], bias) || !pair(a[5], s) || !pair(a[6], p) || !pair(a[7], d) || !pair(a[8], o) ||
        !PyLong_CheckExact(a[9])) NO;
    const int64_t groups = PyLong_AsLongLong(a[9]), N = x->size(0), Cin = x->size(1), Hi = x->size(2), Wi = x->size(3), KH = w->size(2), KW = w->size(3);
    const int64_t Cout = w->size(1) * groups;
    const auto extent = [](int64_t n, int64_t k, int64_t st, int64_t pd, int64_t dl, int64_t op) { return (n - 1) * st - 2 * pd + dl * (k - 1) + op + 1; };
    if (groups < 1 || w->size(0) != Cin || x->numel() < 1 || out->numel() < 1 || !vec_ok(bias, Cout)) NO;
    if (!shape_is(*out, N, Cout, extent(Hi, KH, s[1], p[1], d[1], o[1]), extent(Wi, KW, s[0], p[0], d[0], o[0])) || !env_of(a[0], e)) NO;
    ANSWER(mi_convtranspose2d_f16(ptr(out), ptr(x), ptr(w), ptr(bias), Wi, Hi, Cin, N, KW, KH, Cout, s[0], s[1], p[0], p[1], d[0], d[1], o[0], o[1], groups,
                                         nullptr, 0, e.stream));
}

// ------------------------------------------------------------------------------------------ recorded calls

// A C-ABI call with its arguments in 8-byte slots; `fours` keeps the stride arrays that slots point to.
constexpr int MAX_ARGS = 32;
struct Call;
typedef int (*Invoke)(const uint64_t *);
struct Call {
    Invoke invoke;
    int nargs;
    uint64_t slot[MAX_ARGS];
    std::vector<std::vector<int64_t>> fours;
};
template <typename A> A arg_of(uint64_t s) {
    if constexpr (std::is_pointer_v<A>) return reinterpret_cast<A>((uintptr_t)s);
    else if constexpr (std::is_same_v<A, float>) { float f; std::memcpy(&f, &s, 4); return f; }
    else return (A)(int64_t)s;
}
template <typename A> bool slot_of(PyObject *o, uint64_t &s, Call &c) {
    if constexpr (std::is_same_v<A, float>) {
        double v;
        if (!number(o, v)) return false;
        const float f = (float)v;
        s = 0;
        std::memcpy(&s, &f, 4);
        return true;
    } else if constexpr (std::is_pointer_v<A>) {
        if (o == Py_None) { s = 0; return true; }
        if (PyTuple_CheckExact(o)) {                       // four strides
            std::vector<int64_t> v;
            for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(o); i++) v.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(o, i)));
            c.fours.push_back(std::move(v));
            s = (uint64_t)(uintptr_t)c.fours.back().data();
            return !PyErr_Occurred();
        }
        s = (uint64_t)(uintptr_t)PyLong_AsVoidPtr(o);
        return !PyErr_Occurred();
    } else {
        s = (uint64_t)PyLong_AsLongLong(o);
        return !PyErr_Occurred();
    }
}
template <auto Fn> struct Bound;
template <typename... A, int (*Fn)(A...)> struct Bound<Fn> {
    static constexpr int N = sizeof...(A);
    static_assert(N <= MAX_ARGS, "more arguments than a recorded call holds");
    template <size_t... I> static int go(const uint64_t *s, std::index_sequence<I...>) { return Fn(arg_of<A>(s[I])...); }
    static int invoke(const uint64_t *s) { return go(s, std::index_sequence_for<A...>{}); }
    template <size_t... I> static bool fill_(Call &c, PyObject *args, std::index_sequence<I...>) {
        return (slot_of<A>(PyTuple_GET_ITEM(args, I), c.slot[I], c) && ...);
    }
    static bool fill(Call &c, PyObject *args) {
        c.invoke = invoke;
        c.nargs = N;
        return PyTuple_GET_SIZE(args) == N && fill_(c, args, std::index_sequence_for<A...>{});
    }
};
struct Entry { bool (*fill)(Call &, PyObject *); };
const std::unordered_map<std::string, Entry> &recordable() {          // every call that ends in a stream argument
#define R(f) {#f, {Bound<f>::fill}}
    static const std::unordered_map<std::string, Entry> table = {
        R(mi_gemm_f16), R(mi_gemm_f16_batched), R(mi_gemv_f16), R(mi_ln_gemv_f16), R(mi_ln_gemm_f16), R(mi_gemm_ln_f16), R(mi_gemm_clamp_ln_f16),
        R(mi_rowstats_f16), R(mi_gemm_rowstats_f16), R(mi_lnfold_gemm_f16), R(mi_sdpa_f16), R(mi_conv2d_f16), R(mi_conv2d_nhwc_f16),
        R(mi_conv2d_tokens_f16), R(mi_convtranspose2d_f16), R(mi_transpose_le_f16), R(mi_layernorm_f16), R(mi_softmax_f16), R(mi_scale_f16),
        R(mi_act_f16), R(mi_clamp_f16), R(mi_add_f16), R(mi_kv_append_f16), R(mi_sdpa_append_f16), R(mi_kv_advance), R(mi_kv_len_from_position),
        R(mi_embedding_f16)};
#undef R
    return table;
}
struct Patch { int call, slot, input; int64_t offset; };         // sorted by call
struct CallList {
    std::vector<Call> calls;
    std::vector<Patch> patches;
};
void free_calls(PyObject *cap) { delete static_cast<CallList *>(PyCapsule_GetPointer(cap, "mi_calls")); }

// calls_new([(name, args), ...], [(first address, bytes), ...]) -> capsule, or None where a call cannot be recorded.  The
// ranges are the inputs': a pointer argument that lies in one is issued again relative to that input's new address.
PyObject *calls_new(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(2)
    auto list = std::make_unique<CallList>();
    list->calls.reserve((size_t)PyList_Size(a[0]));
    for (Py_ssize_t i = 0; i < PyList_Size(a[0]); i++) {
        PyObject *rec = PyList_GetItem(a[0], i), *name = PyTuple_GetItem(rec, 0), *args = PyTuple_GetItem(rec, 1);
        if (!name || !args) return nullptr;
        const auto it = recordable().find(PyUnicode_AsUTF8(name));
        if (it == recordable().end()) Py_RETURN_NONE;
        list->calls.emplace_back();
        Call &c = list->calls.back();
        c.fours.reserve(8);                                // slots point into it
        if (PyTuple_GET_SIZE(args) > MAX_ARGS || !it->second.fill(c, args)) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        for (Py_ssize_t r = 0; r < PyList_Size(a[1]); r++) {
            PyObject *range = PyList_GetItem(a[1], r);
            const uint64_t lo = (uint64_t)(uintptr_t)PyLong_AsVoidPtr(PyTuple_GetItem(range, 0)), n = PyLong_AsUnsignedLongLong(PyTuple_GetItem(range, 1));
            for (int s = 0; s < c.nargs - 1; s++) {
                PyObject *v = PyTuple_GET_ITEM(args, s);
                // addresses are far above any extent or stride that an integer argument holds
                if (PyLong_CheckExact(v) && c.slot[s] >= lo && c.slot[s] < lo + n && n)
                    list->patches.push_back({(int)list->calls.size() - 1, s, (int)r, (int64_t)(c.slot[s] - lo)});
            }
        }
        if (PyErr_Occurred()) return nullptr;
    }
    return PyCapsule_New(list.release(), "mi_calls", free_calls);
}

// calls_run(ctx, capsule, inputs tuple) -> True, False (the context is not one this file takes), or the status of the call that was refused
PyObject *calls_run(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(3)
    const CallList *list = static_cast<CallList *>(PyCapsule_GetPointer(a[1], "mi_calls"));
    if (!list) return nullptr;
    Env e;
    if (!env_of(a[0], e)) NO;
    // the addresses first: the list itself stays as it was recorded, so that threads may run it at once
    std::vector<uint64_t> base;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(a[2]); i++) {
        const Tensor *t = tensor(PyTuple_GET_ITEM(a[2], i));
        if (!t) NO;
        base.push_back((uint64_t)(uintptr_t)t->data_ptr());
    }
    const int rc = without_gil([&] {
        auto patch = list->patches.begin();                 // in the order of the calls
        for (size_t i = 0; i < list->calls.size(); i++) {
            const Call &c = list->calls[i];
            uint64_t slot[MAX_ARGS];
            std::memcpy(slot, c.slot, sizeof(uint64_t) * c.nargs);
            for (; patch != list->patches.end() && patch->call == (int)i; ++patch) slot[patch->slot] = base[patch->input] + patch->offset;
            slot[c.nargs - 1] = (uint64_t)(uintptr_t)e.stream;
            const int r = c.invoke(slot);
            if (r != MI_OK) return r;
        }
        return (int)MI_OK;
    });
    if (rc != MI_OK) return PyLong_FromLong(rc);
    Py_RETURN_TRUE;
}

// setup(Workspace type, Ctx type)
PyObject *setup(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    ARITY(2)
    Py_INCREF(a[0]);
    Py_INCREF(a[1]);
    Py_XDECREF(g_workspace_type);
    Py_XDECREF(g_ctx_type);
    g_workspace_type = a[0];
    g_ctx_type = a[1];
    Py_RETURN_NONE;
}

// What torch throws -- an operand without storage, a device that is gone -- ends here: nothing has been enqueued by then (a call
// into the library is the last thing a function does and throws nothing), so the answer is the one that sends the caller to
// the Python form, which meets the same trouble as a Python exception.
typedef PyObject *(*Fast)(PyObject *, PyObject *const *, Py_ssize_t);
template <Fast F, bool TRUTH> PyObject *guarded(PyObject *self, PyObject *const *a, Py_ssize_t nargs) {
    try {
        return F(self, a, nargs);
    } catch (...) {
        PyErr_Clear();
        if (TRUTH) Py_RETURN_FALSE;
        Py_RETURN_NONE;
    }
}

#define M(f) {#f, (PyCFunction)(void (*)(void))(Fast)guarded<f, true>, METH_FASTCALL, nullptr}
#define M_NONE(f) {#f, (PyCFunction)(void (*)(void))(Fast)guarded<f, false>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {M_NONE(setup), M(matmul), M(matmul_rowstats), M(lnfold_matmul), M(ln_matmul), M(layernorm), M(rowstats), M(add), M(sdpa), M(sdpa_append),
                         M(convolution), M(convolutiontranspose), M_NONE(calls_new), M(calls_run), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    s_dev = PyUnicode_InternFromString("dev");
    s_own = PyUnicode_InternFromString("_own");
    s_ws = PyUnicode_InternFromString("ws");
    s_device = PyUnicode_InternFromString("device");
    s_buf = PyUnicode_InternFromString("buf");
    s_off = PyUnicode_InternFromString("off");
    s_scratch = PyUnicode_InternFromString("scratch");
    return PyModule_Create(&module);
}
