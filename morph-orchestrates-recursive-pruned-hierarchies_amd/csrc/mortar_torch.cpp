// Native call layer between torch and libmortar_hip.so: the whole host side of one call of the runtime (checks, output
// and workspace allocation, stream, launches) in one Python call.
//
// A decode-sized MLP is about 10 us of GPU work; the same call assembled in Python (tensor attributes, ctypes argument
// conversion, three allocations) took 30 us of host time and kept the GPU waiting.  Every function returns None for a
// call that it does not cover (another dtype or layout, tensor subclasses, autograd recording): the caller then takes its
// general path, which also words the argument errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <algorithm>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/InferenceMode.h>
#include <c10/hip/HIPStream.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/mortar_hip.h"

namespace {

// One packed matrix as the Python side hands it over (pack.MortarPack.handle): the struct of the C-ABI and the two
// schedules, null until the Python side has built them; then what a re-pack needs (null in a pack that has seen none).
struct PackHandle {
    const mortar_bcsr_t *w;
    const int32_t *sched1, *sched2;
    const int32_t *pos, *src;
    int32_t *status;
    void *workspace;
};

constexpr int DECODE_MAX_ROWS = 64;

const PackHandle *handle_of(PyObject *o) { return static_cast<const PackHandle *>(PyLong_AsVoidPtr(o)); }

// A plain torch.Tensor / Parameter (no subclass that overrides operators) or null.
const at::Tensor *tensor_of(PyObject *o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Truth of any Python object as `if o:` has it (True, 1, numpy.True_, ...); false with the Python error set where it has none.
bool truth(PyObject *o, bool &v) {
    const int t = PyObject_IsTrue(o);
    v = t > 0;
    return t >= 0;
}

PyObject *raise_rc(int rc, const char *what) {
    PyErr_Format(rc == MORTAR_ERR_HIP ? PyExc_RuntimeError : PyExc_ValueError, "%s failed (%d): %s", what, rc, mortar_last_error());
    return nullptr;
}

void *stream_of(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The activation rows of a call: bf16, on the GPU, contiguous, last dimension `d`.
bool is_rows(const at::Tensor &x, int64_t d) {
    return x.is_cuda() && x.scalar_type() == at::kBFloat16 && x.dim() >= 1 && x.size(-1) == d && x.numel() > 0 && x.is_contiguous() &&
           aligned16(x.const_data_ptr());
}

const uint16_t *u16(const at::Tensor &t) { return static_cast<const uint16_t *>(t.const_data_ptr()); }
uint16_t *u16m(const at::Tensor &t) { return static_cast<uint16_t *>(t.data_ptr()); }

at::Tensor new_bf16(const at::Tensor &like, at::IntArrayRef shape) { return at::empty(shape, like.options().requires_grad(false)); }

struct Norm {
    bool on = false;
    const uint16_t *w = nullptr;
    float eps = 0.f;
};

// norm_w: None or a bf16 [d] tensor.  False: not a weight this layer takes.
bool read_norm(PyObject *norm_w, double eps, int64_t d, const at::Tensor &x, Norm &n) {
    n.on = true;
    n.eps = (float)eps;
    if (norm_w == Py_None) return true;
    const at::Tensor *w = tensor_of(norm_w);
    if (!w || w->device() != x.device() || w->scalar_type() != at::kBFloat16 || w->dim() != 1 || w->size(0) != d || !w->is_contiguous() ||
        !aligned16(w->const_data_ptr()))
        return false;
    n.w = u16(*w);
    return true;
}

// gate_up (+ SwiGLU, gates, norm) and down on M rows of x -> y.  The norm is applied inside gate_up where the matrix
// allows it, in its own launch otherwise.
int run_mlp(const PackHandle *gu, const PackHandle *dn, const at::Tensor &x, int64_t M, Norm n, const float *gates, int ncl, uint16_t *y,
            void *st) {
    const int64_t d = (int64_t)gu->w->Cb * 16, f = (int64_t)gu->w->Rb * 8, dy = (int64_t)dn->w->Rb * 16;
    const uint16_t *xp = u16(x);
    at::Tensor xn;
    const bool fused = !n.on || (gu->w->seg_cb >= gu->w->Cb && mortar_norm_fusable(gu->w->Cb));
    at::Tensor h;
    if (M <= DECODE_MAX_ROWS) h = new_bf16(x, {M, f});
    if (!fused && M <= DECODE_MAX_ROWS && !gates) {
        const int rc = mortar_norm_gateup_decode_bf16(gu->w, gu->sched2, xp, M, d, n.w, n.eps, u16m(h), f, st);
        if (rc == MORTAR_OK) return mortar_spmm_bf16(dn->w, dn->sched1, u16(h), M, f, y, dy, st);
        if (rc != MORTAR_NO_KERNEL) return rc;
    }
    if (!fused) {
        xn = new_bf16(x, {M, d});
        const int rc = mortar_rmsnorm_bf16(xp, M, (int32_t)d, d, n.w, n.eps, u16m(xn), d, st);
        if (rc) return rc;
        xp = u16(xn);
        n = Norm{};
    }
    if (M > DECODE_MAX_ROWS) {
        h = at::empty({mortar_mlp_hidden_bytes(M, (int32_t)f)}, x.options().dtype(at::kByte).requires_grad(false));
        return mortar_mlp_bf16(gu->w, gu->sched2, dn->w, dn->sched1, xp, M, d, n.on, n.w, n.eps, gates, ncl, h.data_ptr(), y, dy, 0, st);
    }
    int rc = n.on ? mortar_norm_gateup_swiglu_bf16(gu->w, gu->sched2, xp, M, d, n.w, n.eps, u16m(h), f, gates, ncl, nullptr, nullptr, st)
                  : mortar_gateup_swiglu_bf16(gu->w, gu->sched2, xp, M, d, u16m(h), f, gates, ncl, nullptr, nullptr, st);
    if (rc == MORTAR_OK) rc = mortar_spmm_bf16(dn->w, dn->sched1, u16(h), M, f, y, dy, st);
    return rc;
}

// mlp(x, gate_up handle, down handle, decode, norm, norm_w, eps, gates) -> y: the carved MLP on the rows of x.
// gates: None or fp32 [..., n_clusters], one row per row of x.  decode: x [B, ...] is one row per stream and y is [B, 1, d] whatever autograd records (MortarDecodeMLP); otherwise y
// has the shape of x and a call that autograd would record is declined.
PyObject *py_mlp(PyObject *, PyObject *const *a, Py_ssize_t na) {
    if (na != 8) {
        PyErr_SetString(PyExc_TypeError, "mlp: 8 arguments");
        return nullptr;
    }
    const at::Tensor *xt = tensor_of(a[0]);
    const PackHandle *gu = handle_of(a[1]), *dn = handle_of(a[2]);
    if (PyErr_Occurred()) return nullptr;
    bool decode, norm;
    const double eps = PyFloat_AsDouble(a[6]);
    if (PyErr_Occurred() || !truth(a[3], decode) || !truth(a[4], norm)) return nullptr;
    if (!xt || !gu || !dn || !gu->sched2 || !dn->sched1) Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int64_t d = (int64_t)gu->w->Cb * 16;
    if (!is_rows(x, d) || (!decode && x.requires_grad() && c10::GradMode::is_enabled())) Py_RETURN_NONE;
    const int64_t M = x.numel() / d;
    if (decode && x.size(0) != M) Py_RETURN_NONE;
    Norm n;
    if (norm && !read_norm(a[5], eps, d, x, n)) Py_RETURN_NONE;
    const float *gates = nullptr;
    int64_t ncl = 0;
    if (a[7] != Py_None) {
        const at::Tensor *gt = tensor_of(a[7]);
        const int64_t f = (int64_t)gu->w->Rb * 8;
        if (!gt || gt->scalar_type() != at::kFloat || gt->device() != x.device() || gt->dim() < 1 || !gt->is_contiguous()) Py_RETURN_NONE;
        ncl = gt->size(-1);
        if (ncl <= 0 || gt->numel() != M * ncl || f % ncl || (f / ncl) % 4) Py_RETURN_NONE;
        gates = static_cast<const float *>(gt->const_data_ptr());
    }
    const int64_t dy = (int64_t)dn->w->Rb * 16;
    const c10::DeviceGuard guard(x.device());
    at::Tensor y;
    if (decode) {
        y = new_bf16(x, {M, 1, dy});
    } else {
        at::DimVector shape(x.sizes());
        shape.back() = dy;
        y = new_bf16(x, shape);
    }
    const int rc = run_mlp(gu, dn, x, M, n, gates, (int)ncl, u16m(y), stream_of(x));
    if (rc) return raise_rc(rc, "mortar_mlp");
    return THPVariable_Wrap(std::move(y));
}

// ---- router ------------------------------------------------------------------------------------------------------

// The parameters of a TileRouter, looked up in its modules' dictionaries at every call (a parameter that was replaced or
// moved is then seen as it is).
struct RouterParams {
    const float *wq, *iter_vec, *ln_w, *ln_b, *ka, *kb, *bias;
    int32_t nsk, n;
};

enum { N_WEIGHT, N_BIAS, N_KEYS_A, N_KEYS_B, N_GROUP_BIAS, N_ITER, N_NAMES };
PyObject *g_names[N_NAMES];

const float *f32_param(PyObject *dict, int name, const at::Tensor &x, at::IntArrayRef shape) {
    PyObject *o = PyDict_GetItem(dict, g_names[name]);
    const at::Tensor *t = o ? tensor_of(o) : nullptr;
    if (!t || t->scalar_type() != at::kFloat || t->device() != x.device() || t->sizes() != shape || !t->is_contiguous() ||
        !aligned16(t->const_data_ptr()))
        return nullptr;
    return static_cast<const float *>(t->const_data_ptr());
}

// own / proj / norm: the `_parameters` dictionaries of the router, its query_proj and its query_norm.
bool read_router(PyObject *own, PyObject *proj, PyObject *norm, int64_t it, int64_t n_iters, int64_t nsk, int64_t n, int64_t d,
                 const at::Tensor &x, RouterParams &r) {
    if (!PyDict_Check(own) || !PyDict_Check(proj) || !PyDict_Check(norm)) return false;
    r.wq = f32_param(proj, N_WEIGHT, x, {d, d});
    r.ln_w = f32_param(norm, N_WEIGHT, x, {d});
    r.ln_b = f32_param(norm, N_BIAS, x, {d});
    r.ka = f32_param(own, N_KEYS_A, x, {nsk, d / 2});
    r.kb = f32_param(own, N_KEYS_B, x, {nsk, d / 2});
    r.bias = f32_param(own, N_GROUP_BIAS, x, {n});
    const float *emb = f32_param(own, N_ITER, x, {n_iters, d});
    if (!r.wq || !r.ln_w || !r.ln_b || !r.ka || !r.kb || !r.bias || !emb) return false;
    it = it < 0 ? 0 : it >= n_iters ? n_iters - 1 : it;
    r.iter_vec = emb + it * d;
    r.nsk = (int32_t)nsk;
    r.n = (int32_t)n;
    return aligned16(r.iter_vec);
}

// routed_decode(x, gate_up handle, down handle, norm_w, eps, own, proj, norm, shape, ln_eps, iter_idx) -> y [B, 1, d]:
// RMSNorm, router, gated gate_up, down for up to 64 single-token rows.  shape = (n_iters, n_sub_keys, n_groups, k).
PyObject *py_routed_decode(PyObject *, PyObject *const *a, Py_ssize_t na) {
    if (na != 11 || !PyTuple_Check(a[8]) || PyTuple_GET_SIZE(a[8]) != 4) {
        PyErr_SetString(PyExc_TypeError, "routed_decode: 11 arguments");
        return nullptr;
    }
    const at::Tensor *xt = tensor_of(a[0]);
    const PackHandle *gu = handle_of(a[1]), *dn = handle_of(a[2]);
    int64_t sh[4];
    for (int i = 0; i < 4; ++i) sh[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(a[8], i));
    const double eps = PyFloat_AsDouble(a[4]), ln_eps = PyFloat_AsDouble(a[9]);
    const int64_t it = PyLong_AsLongLong(a[10]);
    if (PyErr_Occurred()) return nullptr;
    if (!xt || !gu || !dn || !gu->sched2 || !dn->sched1) Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int64_t d = (int64_t)gu->w->Cb * 16, f = (int64_t)gu->w->Rb * 8, n = sh[2];
    if (!is_rows(x, d) || d % 8 || d > 8192 || sh[1] <= 0 || sh[1] * sh[1] > 2048 || n <= 0 || n > 1024 || f % n || (f / n) % 4) Py_RETURN_NONE;
    const int64_t M = x.numel() / d;
    if (M > DECODE_MAX_ROWS || x.size(0) != M) Py_RETURN_NONE;
    Norm nm;
    RouterParams r;
    if (!read_norm(a[3], eps, d, x, nm) || !read_router(a[5], a[6], a[7], it, sh[0], sh[1], n, d, x, r)) Py_RETURN_NONE;
    const c10::DeviceGuard guard(x.device());
    void *st = stream_of(x);
    const at::Tensor xn = new_bf16(x, {M, d});
    // one workspace: the projected queries, then the gates
    const at::Tensor ws = at::empty({M * (d + n)}, x.options().dtype(at::kFloat).requires_grad(false));
    float *qv = static_cast<float *>(ws.data_ptr()), *gates = qv + M * d;
    at::Tensor y = new_bf16(x, {M, 1, (int64_t)dn->w->Rb * 16});
    int rc = mortar_norm_router_bf16(u16(x), M, (int32_t)d, d, nm.w, nm.eps, u16m(xn), r.wq, r.iter_vec, r.ln_w, r.ln_b, (float)ln_eps, r.ka, r.kb,
                                     r.nsk, r.bias, r.n, (int32_t)sh[3], qv, nullptr, gates, nullptr, st);
    if (rc == MORTAR_OK) rc = run_mlp(gu, dn, xn, M, Norm{}, gates, (int)n, u16m(y), st);
    if (rc) return raise_rc(rc, "mortar_routed_decode");
    return THPVariable_Wrap(std::move(y));
}

// route(x, own, proj, norm, shape, ln_eps, iter_idx, ema, alpha, coeff) -> (gates [M, n], active [M, n], aux): the router of
// the M rows of x, without autograd.  With ema (the load statistics buffer, fp32 [n]) the statistics are updated in place
// and aux is the load-balance loss; with ema = None aux is None.  The in-place update counts as one for autograd and others
// who look at the version of the buffer.
PyObject *py_route(PyObject *, PyObject *const *a, Py_ssize_t na) {
    if (na != 10 || !PyTuple_Check(a[4]) || PyTuple_GET_SIZE(a[4]) != 4) {
        PyErr_SetString(PyExc_TypeError, "route: 10 arguments");
        return nullptr;
    }
    int64_t sh[4];
    for (int i = 0; i < 4; ++i) sh[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(a[4], i));
    const double ln_eps = PyFloat_AsDouble(a[5]), alpha = PyFloat_AsDouble(a[8]), coeff = PyFloat_AsDouble(a[9]);
    const int64_t it = PyLong_AsLongLong(a[6]), nsk = sh[1], n = sh[2];
    if (PyErr_Occurred()) return nullptr;
    const at::Tensor *xt = tensor_of(a[0]);
    if (!xt || c10::GradMode::is_enabled() || xt->dim() < 1) Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int64_t d = x.size(-1);
    if (d % 8 || d > 8192 || nsk <= 0 || n <= 0 || n > 1024 || !is_rows(x, d)) Py_RETURN_NONE;
    const int64_t M = x.numel() / d;
    const bool small = M <= DECODE_MAX_ROWS;
    if (nsk * nsk > (small ? 2048 : std::max<int64_t>(1024, n))) Py_RETURN_NONE;
    RouterParams r;
    if (!read_router(a[1], a[2], a[3], it, sh[0], nsk, n, d, x, r)) Py_RETURN_NONE;
    const at::Tensor *ema = a[7] == Py_None ? nullptr : tensor_of(a[7]);
    if (a[7] != Py_None && (!ema || ema->scalar_type() != at::kFloat || ema->device() != x.device() || ema->dim() != 1 || ema->size(0) != n ||
                            !ema->is_contiguous() || (ema->is_inference() && !c10::InferenceMode::is_enabled())))
        Py_RETURN_NONE;          // (an inference tensor outside inference mode: torch's in-place operators word that error)
    const c10::DeviceGuard guard(x.device());
    void *st = stream_of(x);
    const auto f32 = x.options().dtype(at::kFloat).requires_grad(false);
    at::Tensor gates = at::empty({M, n}, f32), active = at::empty({M, n}, f32.dtype(at::kByte)), aux;
    float *gp = static_cast<float *>(gates.data_ptr());
    uint8_t *ap = static_cast<uint8_t *>(active.data_ptr());
    const at::Tensor qvt = at::empty({M, d}, f32);
    float *qv = static_cast<float *>(qvt.data_ptr());
    int rc;
    if (small) {
        rc = mortar_router_bf16(u16(x), 0, M, (int32_t)d, d, r.wq, r.iter_vec, r.ln_w, r.ln_b, (float)ln_eps, r.ka, r.kb, r.nsk, r.bias, r.n,
                                (int32_t)sh[3], qv, nullptr, gp, ap, st);
    } else {
        rc = mortar_router_project_bf16(u16(x), M, (int32_t)d, d, r.wq, (int32_t)d, qv, d, st);
        if (rc == MORTAR_OK)
            rc = mortar_router_tail_f32(qv, M, (int32_t)d, d, r.iter_vec, r.ln_w, r.ln_b, (float)ln_eps, r.ka, r.kb, r.nsk, r.bias, r.n,
                                        (int32_t)sh[3], nullptr, gp, ap, st);
    }
    if (rc == MORTAR_OK && ema) {
        aux = at::empty({}, f32);
        const at::Tensor ws = at::empty({mortar_router_stats_workspace_bytes(M, r.n)}, f32.dtype(at::kByte));
        rc = mortar_router_stats(gp, M, r.n, (float)alpha, (float)(1.0 - alpha), (float)coeff, static_cast<float *>(ema->data_ptr()),
                                 static_cast<float *>(aux.data_ptr()), ws.data_ptr(), st);
        if (rc == MORTAR_OK && !ema->is_inference()) ema->unsafeGetTensorImpl()->bump_version();      // written through its address
    }
    if (rc) return raise_rc(rc, "mortar_route");
    PyObject *g = THPVariable_Wrap(std::move(gates)), *ac = THPVariable_Wrap(std::move(active));
    PyObject *au = Py_None;
    if (aux.defined()) au = THPVariable_Wrap(std::move(aux));
    else Py_INCREF(Py_None);
    return Py_BuildValue("(NNN)", g, ac, au);
}

// Optional integer flags [B, >= n] of a decode product.  False: not flags this layer takes.
bool read_flags(PyObject *o, const at::Tensor &x, int64_t B, int64_t n, const int32_t *&p, int64_t &ld) {
    p = nullptr;
    ld = 0;
    if (o == Py_None) return true;
    const at::Tensor *t = tensor_of(o);
    if (!t || t->scalar_type() != at::kInt || t->device() != x.device() || t->dim() != 2 || t->size(0) != B || t->size(1) < n || t->stride(1) != 1)
        return false;
    p = static_cast<const int32_t *>(t->const_data_ptr());
    ld = t->stride(0);
    return true;
}

// gemv_f32(x, handle, scale, swiglu_x, swiglu_out, gates, row_act, col_act) -> y fp32 [B, out]: the decode product in the
// reference engine's arithmetic for a matrix with one scale.
PyObject *py_gemv_f32(PyObject *, PyObject *const *a, Py_ssize_t na) {
    if (na != 8) {
        PyErr_SetString(PyExc_TypeError, "gemv_f32: 8 arguments");
        return nullptr;
    }
    const at::Tensor *xt = tensor_of(a[0]), *sc = tensor_of(a[2]);
    const PackHandle *h = handle_of(a[1]);
    bool swx, swo;
    if (PyErr_Occurred() || !truth(a[3], swx) || !truth(a[4], swo)) return nullptr;
    if (!xt || !sc || !h || sc->numel() != 1 || sc->scalar_type() != at::kFloat) Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int64_t K = (int64_t)h->w->Cb * 16, nout = (int64_t)h->w->Rb * (swo ? 8 : 16);
    if (!x.is_cuda() || sc->device() != x.device() || x.scalar_type() != at::kFloat || x.dim() != 2 || x.size(1) != K * (swx ? 2 : 1) ||
        !x.is_contiguous() || !aligned16(x.const_data_ptr()) || (swo && (h->w->Rb & 1)))
        Py_RETURN_NONE;
    const int64_t B = x.size(0);
    if (B < 1 || B > DECODE_MAX_ROWS || !mortar_gemv_f32_one_better(h->w, swo, (int32_t)B)) Py_RETURN_NONE;
    const float *gates = nullptr;
    int64_t ncl = 0, ldg = 0;
    if (a[5] != Py_None) {
        const at::Tensor *gt = tensor_of(a[5]);
        if (!gt || !swo || gt->scalar_type() != at::kFloat || gt->device() != x.device() || gt->dim() != 2 || gt->size(0) != B || gt->stride(1) != 1)
            Py_RETURN_NONE;
        ncl = gt->size(1);
        ldg = gt->stride(0);
        if (ncl <= 0 || nout % ncl || (nout / ncl) % 4) Py_RETURN_NONE;
        gates = static_cast<const float *>(gt->const_data_ptr());
    }
    const int32_t *ra, *ca;
    int64_t ldr, ldc;
    if (!read_flags(a[6], x, B, h->w->Rb, ra, ldr) || !read_flags(a[7], x, B, h->w->Cb, ca, ldc)) Py_RETURN_NONE;
    const c10::DeviceGuard guard(x.device());
    at::Tensor y = at::empty({B, nout}, x.options().requires_grad(false));
    const int rc = mortar_gemv_f32_one(h->w, static_cast<const float *>(sc->const_data_ptr()), swo, swx, static_cast<const float *>(x.const_data_ptr()),
                                       (int32_t)B, x.size(1), static_cast<float *>(y.data_ptr()), nout, gates, (int32_t)ncl, ldg, ra, ldr, ca, ldc,
                                       stream_of(x));
    if (rc == MORTAR_NO_KERNEL) Py_RETURN_NONE;
    if (rc) return raise_rc(rc, "mortar_gemv_f32");
    return THPVariable_Wrap(std::move(y));
}

// ---- training step of the MLP ------------------------------------------------------------------------------------

// Block values [nnz, 16, 16] of a matrix, bf16 or fp32.
bool is_values(const at::Tensor &v, const mortar_bcsr_t *w, const at::Tensor &x) {
    return v.device() == x.device() && (v.scalar_type() == at::kBFloat16 || v.scalar_type() == at::kFloat) && v.dim() == 3 && v.size(0) == w->nnz &&
           v.size(1) == 16 && v.size(2) == 16 && v.is_contiguous() && aligned16(v.const_data_ptr());
}

// A matrix as the products of a training step take it: the step re-packs it, so that its scale is one at every replay of a captured
// step as well.
mortar_bcsr_t step_form(const PackHandle *h) {
    mortar_bcsr_t w = *h->w;
    if (w.one_scale) w.one_scale = 2;
    return w;
}

bool repackable(const PackHandle *h) { return h->pos && h->status && h->workspace && h->sched1; }

mortar_repack_t repack_of(const PackHandle *h, const PackHandle *t, const at::Tensor &v, double threshold, const at::Tensor &scale) {
    mortar_repack_t r{};
    r.W = h->w; r.pos = h->pos; r.status = h->status; r.workspace = h->workspace; r.scale_out = static_cast<float *>(scale.data_ptr());
    if (t) { r.Wt = t->w; r.pos_t = t->pos; r.src_t = t->src; r.status_t = t->status; }
    r.values = v.const_data_ptr();
    r.values_f32 = v.scalar_type() == at::kFloat;
    r.threshold = (float)threshold;
    return r;
}

// train_forward(x, gate_up values, down values, gate_up, its W^T or 0, down, its W^T or 0, thresholds of the two) -> (y, gu, h,
// scale of gate_up, of down): the re-pack of both matrices and the transposes named, then gate_up, SwiGLU and down on the rows of x.  No
// autograd of its own.
PyObject *py_train_forward(PyObject *, PyObject *const *a, Py_ssize_t na) {
    if (na != 9) {
        PyErr_SetString(PyExc_TypeError, "train_forward: 9 arguments");
        return nullptr;
    }
    const at::Tensor *xt = tensor_of(a[0]), *vg = tensor_of(a[1]), *vd = tensor_of(a[2]);
    const PackHandle *gu = handle_of(a[3]), *gut = handle_of(a[4]), *dn = handle_of(a[5]), *dnt = handle_of(a[6]);
    if (PyErr_Occurred()) return nullptr;
    const double tg = PyFloat_AsDouble(a[7]), td = PyFloat_AsDouble(a[8]);
    if (PyErr_Occurred()) return nullptr;
    if (!xt || !vg || !vd || !gu || !dn || !repackable(gu) || !repackable(dn) || (gut && !(repackable(gut) && gut->src)) ||
        (dnt && !(repackable(dnt) && dnt->src)))
        Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int64_t d = (int64_t)gu->w->Cb * 16, f2 = (int64_t)gu->w->Rb * 16, f = (int64_t)dn->w->Cb * 16, dy = (int64_t)dn->w->Rb * 16;
    if (x.dim() != 2 || !is_rows(x, d) || f2 != 2 * f || !is_values(*vg, gu->w, x) || !is_values(*vd, dn->w, x)) Py_RETURN_NONE;
    const int64_t M = x.size(0);
    const c10::DeviceGuard guard(x.device());
    void *st = stream_of(x);
    const auto f32 = x.options().dtype(at::kFloat).requires_grad(false);
    at::Tensor sg = at::empty({1}, f32), sd = at::empty({1}, f32);
    const mortar_repack_t re[2] = {repack_of(gu, gut, *vg, tg, sg), repack_of(dn, dnt, *vd, td, sd)};
    at::Tensor g = new_bf16(x, {M, f2}), h = new_bf16(x, {M, f}), y = new_bf16(x, {M, dy});
    const mortar_bcsr_t wg = step_form(gu), wd = step_form(dn);
    int rc = mortar_requantize_pairs(re, 2, st);
    if (rc == MORTAR_OK) rc = mortar_spmm_bf16(&wg, gu->sched1, u16(x), M, d, u16m(g), f2, st);
    if (rc == MORTAR_OK) rc = mortar_swiglu_bf16(u16(g), f2, M, (int32_t)f, u16m(h), f, st);
    if (rc == MORTAR_OK) rc = mortar_spmm_bf16(&wd, dn->sched1, u16(h), M, f, u16m(y), dy, st);
    if (rc) return raise_rc(rc, "mortar_train_forward");
    return Py_BuildValue("(NNNNN)", THPVariable_Wrap(std::move(y)), THPVariable_Wrap(std::move(g)), THPVariable_Wrap(std::move(h)),
                         THPVariable_Wrap(std::move(sg)), THPVariable_Wrap(std::move(sd)));
}

// A weight gradient's plan as the Python side hands it over: (address, workgroups, blocks per wave), or None / no need.
struct SddPlan {
    const int32_t *plan = nullptr;
    int32_t n_wg = 0, nb = 0;
};
bool read_plan(PyObject *o, SddPlan &p) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) < 3) return false;
    p.plan = static_cast<const int32_t *>(PyLong_AsVoidPtr(PyTuple_GET_ITEM(o, 0)));
    p.n_wg = (int32_t)PyLong_AsLong(PyTuple_GET_ITEM(o, 1));
    p.nb = (int32_t)PyLong_AsLong(PyTuple_GET_ITEM(o, 2));
    return !PyErr_Occurred() && p.plan;
}

// out[j] = a[:, rows of block j]^T b[:, columns of block j] on a topology of Rb x Cb block-rows and -columns.
int run_sdd(const SddPlan &p, int32_t Rb, int32_t Cb, int64_t nnz, const at::Tensor &a, const at::Tensor &b, at::Tensor &out, void *st) {
    const int64_t M = a.size(0), ws = mortar_sdd_workspace_bytes(p.n_wg, (int32_t)nnz, p.nb, M);
    if (ws < 0) return (int)ws;
    const at::Tensor acc = at::empty({ws}, a.options().dtype(at::kByte).requires_grad(false));
    out = new_bf16(a, {nnz, 16, 16});
    return mortar_sdd_bf16(p.plan, p.n_wg, p.nb, Rb, Cb, (int32_t)nnz, u16(a), a.stride(0), u16(b), b.stride(0), M, static_cast<float *>(acc.data_ptr()),
                           u16m(out), st);
}

PyObject *wrap_or_none(at::Tensor &t) {
    if (t.defined()) return THPVariable_Wrap(std::move(t));
    Py_RETURN_NONE;
}

// train_backward(dy, x, gu, h, gate_up, its W^T or 0, down, its W^T or 0, plan of d(gate_up) or None, plan of d(down) or None) ->
// (dx, d gate_up, d down): dx where gate_up's W^T is given, the weight gradients where their plans are; None elsewhere.
PyObject *py_train_backward(PyObject *, PyObject *const *a, Py_ssize_t na) {
    if (na != 10) {
        PyErr_SetString(PyExc_TypeError, "train_backward: 10 arguments");
        return nullptr;
    }
    const at::Tensor *t[4];
    for (int i = 0; i < 4; ++i) t[i] = tensor_of(a[i]);
    const PackHandle *gu = handle_of(a[4]), *gut = handle_of(a[5]), *dn = handle_of(a[6]), *dnt = handle_of(a[7]);
    if (PyErr_Occurred()) return nullptr;
    if (!t[0] || !t[1] || !t[2] || !t[3] || !gu || !dn) Py_RETURN_NONE;
    const at::Tensor &dy = *t[0], &x = *t[1], &g = *t[2], &h = *t[3];
    const int64_t d = (int64_t)gu->w->Cb * 16, f2 = (int64_t)gu->w->Rb * 16, f = (int64_t)dn->w->Cb * 16, dd = (int64_t)dn->w->Rb * 16;
    for (int i = 0; i < 4; ++i)
        if (t[i]->dim() != 2 || !is_rows(*t[i], i == 0 ? dd : i == 1 ? d : i == 2 ? f2 : f) || t[i]->size(0) != x.size(0) || t[i]->device() != x.device())
            Py_RETURN_NONE;
    SddPlan pg, pd;
    const bool need_gu = a[8] != Py_None, need_dn = a[9] != Py_None;
    if ((need_gu && !read_plan(a[8], pg)) || (need_dn && !read_plan(a[9], pd))) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    if ((gut && !gut->sched1) || ((gut || need_gu) && (!dnt || !dnt->sched1))) Py_RETURN_NONE;
    const int64_t M = x.size(0);
    const c10::DeviceGuard guard(x.device());
    void *st = stream_of(x);
    at::Tensor dx, dgu, ddn;
    int rc = MORTAR_OK;
    if (need_dn) rc = run_sdd(pd, dn->w->Rb, dn->w->Cb, dn->w->nnz, dy, h, ddn, st);
    if (rc == MORTAR_OK && (gut || need_gu)) {
        const at::Tensor dh = new_bf16(x, {M, f}), dg = new_bf16(x, {M, f2});
        const mortar_bcsr_t wdt = step_form(dnt);
        rc = mortar_spmm_bf16(&wdt, dnt->sched1, u16(dy), M, dd, u16m(dh), f, st);
        if (rc == MORTAR_OK) rc = mortar_swiglu_backward_bf16(u16(g), f2, u16(dh), f, M, (int32_t)f, u16m(dg), f2, st);
        if (rc == MORTAR_OK && need_gu) rc = run_sdd(pg, gu->w->Rb, gu->w->Cb, gu->w->nnz, dg, x, dgu, st);
        if (rc == MORTAR_OK && gut) {
            dx = new_bf16(x, {M, d});
            const mortar_bcsr_t wgt = step_form(gut);
            rc = mortar_spmm_bf16(&wgt, gut->sched1, u16(dg), M, f2, u16m(dx), d, st);
        }
    }
    if (rc) return raise_rc(rc, "mortar_train_backward");
    PyObject *r0 = wrap_or_none(dx), *r1 = wrap_or_none(dgu), *r2 = wrap_or_none(ddn);
    return Py_BuildValue("(NNN)", r0, r1, r2);
}

// ---- the product over stored block values as one autograd node ---------------------------------------------------

// pack.BcsrTopology as the Python side hands it over; src: of a transposed topology, the block of W behind each block.
struct TopologyHandle {
    const int32_t *row_ptr;
    const int16_t *col;
    const int32_t *seg_ptr, *src;
    int32_t Rb, Cb;
    int64_t nnz;
};

// An owned Python reference that may be dropped on a thread that does not hold the interpreter.
struct PyOwned {
    PyObject *o = nullptr;
    explicit PyOwned(PyObject *p) : o(p) {}
    PyOwned(const PyOwned &) = delete;
    PyOwned &operator=(const PyOwned &) = delete;
    ~PyOwned() {
        if (!o || !Py_IsInitialized()) return;
        const PyGILState_STATE g = PyGILState_Ensure();
        Py_DECREF(o);
        PyGILState_Release(g);
    }
};

// Nothing rides on the tensor that a kernel launched on its address would pass by: no subclass, functorch wrapper, lazy view or
// forward gradient.
c10::DispatchKeySet riders() {
    using K = c10::DispatchKey;
    return c10::DispatchKeySet({K::Python, K::PythonTLSSnapshot, K::FuncTorchGradWrapper, K::FuncTorchBatched, K::FuncTorchDynamicLayerFrontMode,
                                K::FuncTorchDynamicLayerBackMode, K::Batched, K::Functionalize, K::Conjugate, K::Negative, K::ZeroTensor, K::Tracer});
}
bool is_bare(const at::Tensor &t) {
    return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(riders()) && !t._fw_grad(0).defined();
}
// No transform, mode or tracer looks on.
bool nothing_looks_on() {
    return !c10::impl::tls_local_dispatch_key_set().included_.has_any(riders()) && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing();
}

struct DdsShape {
    int64_t s0, s1;
    bool tb;
};

// Operands that the native product takes: x [M, s0] bf16 rows and data [nnz, 16, 16] bf16.
bool dds_covers(const at::Tensor &x, const at::Tensor &data, DdsShape s) {
    return x.scalar_type() == at::kBFloat16 && x.dim() == 2 && x.size(0) > 0 && x.size(0) <= (1 << 30) && x.size(1) == s.s0 && s.s0 > 0 && s.s1 > 0 &&
           x.stride(1) == 1 && x.stride(0) >= s.s0 && x.stride(0) % 8 == 0 && aligned16(x.const_data_ptr()) && data.scalar_type() == at::kBFloat16 &&
           data.dim() == 3 && data.size(0) > 0 && data.size(1) == 16 && data.size(2) == 16 && data.is_contiguous() && aligned16(data.const_data_ptr()) &&
           data.device() == x.device();
}

// Calls one of the Python side's look-ups; the result holds what the launches read until they are enqueued.  Needs the interpreter.
PyObject *look_up(PyObject *fn, const at::Tensor &off, const at::Tensor &col, const at::Tensor &data, int64_t out_f, int64_t in_f, PyObject *last) {
    return PyObject_CallFunction(fn, "NNNLLN", THPVariable_Wrap(off), THPVariable_Wrap(col), THPVariable_Wrap(data), (long long)out_f, (long long)in_f, last);
}

// y = x W^T (tb) or x W on a looked-up topology; undefined, with nothing launched, where the entry point refuses the call.
at::Tensor run_dds(const TopologyHandle *t, const at::Tensor &x, const at::Tensor &data) {
    const c10::DeviceGuard guard(x.device());
    void *st = stream_of(x);
    const int64_t M = x.size(0), n = (int64_t)t->Rb * 16;
    at::Tensor w = data;
    int rc = MORTAR_OK;
    if (t->src) {
        w = new_bf16(data, data.sizes());
        rc = mortar_transpose_blocks_bf16(u16(data), t->src, t->nnz, u16m(w), st);
    }
    at::Tensor y = new_bf16(x, {M, n});
    if (rc == MORTAR_OK)
        rc = mortar_dds_values_bf16(t->row_ptr, t->col, t->seg_ptr, u16(w), t->Rb, t->Cb, t->nnz, u16(x), M, x.stride(0), u16m(y), n, st);
    TORCH_CHECK(rc == MORTAR_OK, "mortar_dds_values_bf16 failed (", rc, "): ", mortar_last_error());
    return y;
}

// The look-ups of stk.py, owned by the node that will use them in its backward.
struct LookUps : torch::CustomClassHolder {
    PyOwned topology, plan;
    LookUps(PyObject *t, PyObject *p) : topology(Py_NewRef(t)), plan(Py_NewRef(p)) {}
};
struct DdsCall {
    const TopologyHandle *topo;            // of the forward product: not kept
    PyObject *find_topology, *find_plan;
};

at::Tensor call_op(const char *name, std::vector<c10::IValue> args) {
    const auto op = c10::Dispatcher::singleton().findSchemaOrThrow(name, "");
    torch::jit::Stack stack(std::move(args));
    op.callBoxed(&stack);
    return stack.at(0).toTensor();
}

struct DdsFn : public torch::autograd::Function<DdsFn> {
    static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &x, const at::Tensor &data, const at::Tensor &off, const at::Tensor &row,
                              const at::Tensor &col, const at::Tensor &off_t, const at::Tensor &col_t, const at::Tensor &blk_t, DdsShape s, DdsCall c) {
        ctx->save_for_backward({x, data, off, row, col, off_t, col_t, blk_t});
        ctx->saved_data["s0"] = s.s0;
        ctx->saved_data["s1"] = s.s1;
        ctx->saved_data["tb"] = s.tb;
        ctx->saved_data["find"] = c10::IValue::make_capsule(c10::make_intrusive<LookUps>(c.find_topology, c.find_plan));
        return run_dds(c.topo, x, data);
    }

    // dx = dy (W if tb else W^T): another dds; ddata = (dy^T x if tb else x^T dy) on the topology (reference: custom_ops.py:99-136).
    // Gradients of other kinds, and those that autograd records again, go through the operators.
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto v = ctx->get_saved_variables();
        const at::Tensor &x = v[0], &data = v[1], &off = v[2], &col = v[4];
        const DdsShape s{ctx->saved_data["s0"].toInt(), ctx->saved_data["s1"].toInt(), ctx->saved_data["tb"].toBool()};
        const auto look = c10::static_intrusive_pointer_cast<LookUps>(ctx->saved_data["find"].toCapsule());
        torch::autograd::variable_list out(10);
        if (!grads[0].defined()) return out;
        const at::Tensor dy = grads[0].contiguous();
        const bool native = !c10::GradMode::is_enabled() && nothing_looks_on() && is_bare(dy) && is_bare(x) && is_bare(data) &&
                            dds_covers(dy, data, {s.s1, s.s0, !s.tb}) && dds_covers(x, data, s) && dy.size(0) == x.size(0) && dy.device() == x.device();
        if (ctx->needs_input_grad(0)) {
            if (native) {
                const PyOwned held(find(look->topology.o, off, col, data, s.tb ? s.s1 : s.s0, s.tb ? s.s0 : s.s1, s.tb ? Py_True : Py_False, -1));
                out[0] = run_dds(topology_of(held.o), dy, data);
            } else {
                out[0] = call_op("mortar_amd::dds", {dy, data, off, v[3], col, v[5], v[6], v[7], s.s1, s.s0, !s.tb});
            }
        }
        if (ctx->needs_input_grad(1)) {
            const at::Tensor &a = s.tb ? dy : x, &b = s.tb ? x : dy;
            if (native) {
                const int64_t out_f = s.tb ? s.s1 : s.s0, in_f = s.tb ? s.s0 : s.s1;
                const PyOwned held(find(look->plan.o, off, col, data, out_f, in_f, nullptr, dy.size(0)));
                SddPlan p;
                {
                    const PyGILState_STATE g = PyGILState_Ensure();
                    const bool ok = read_plan(held.o, p);
                    PyErr_Clear();
                    PyGILState_Release(g);
                    TORCH_CHECK(ok, "stk_dds: no plan for the weight gradient");
                }
                const c10::DeviceGuard guard(x.device());
                const int rc = run_sdd(p, (int32_t)(out_f / 16), (int32_t)(in_f / 16), data.size(0), a, b, out[1], stream_of(x));
                TORCH_CHECK(rc == MORTAR_OK, "mortar_sdd_bf16 failed (", rc, "): ", mortar_last_error());
            } else {
                out[1] = call_op("mortar_amd::sdd_at_b", {a, b, data, off, v[3], col});
                if (out[1].scalar_type() != data.scalar_type()) out[1] = out[1].to(data.scalar_type());
            }
        }
        return out;
    }

    static const TopologyHandle *topology_of(PyObject *held) {
        const PyGILState_STATE g = PyGILState_Ensure();
        const auto *t = static_cast<const TopologyHandle *>(PyLong_AsVoidPtr(PyTuple_GET_ITEM(held, 0)));
        PyGILState_Release(g);
        return t;
    }

    // A look-up from the backward's thread; its Python errors travel with the autograd engine's.
    static PyObject *find(PyObject *fn, const at::Tensor &off, const at::Tensor &col, const at::Tensor &data, int64_t out_f, int64_t in_f, PyObject *flag,
                          int64_t number) {
        const PyGILState_STATE g = PyGILState_Ensure();
        if (flag) Py_INCREF(flag);
        PyObject *r = look_up(fn, off, col, data, out_f, in_f, flag ? flag : PyLong_FromLongLong(number));
        if (!r) {
            python_error err;
            err.persist();
            PyGILState_Release(g);
            throw err;
        }
        PyGILState_Release(g);
        return r;
    }
};

// dds(topology look-up, plan look-up, lhs, data, offsets, row_indices, column_indices, offsets_t, column_indices_t, block_offsets_t, shape0,
// shape1, transpose_b) -> y with its autograd node, or None: stk_dds on plain bf16 tensors.
PyObject *py_dds(PyObject *, PyObject *const *a, Py_ssize_t na) {
    if (na != 13) {
        PyErr_SetString(PyExc_TypeError, "dds: 13 arguments");
        return nullptr;
    }
    const at::Tensor *t[8];
    for (int i = 0; i < 8; ++i)
        if (!(t[i] = tensor_of(a[2 + i]))) Py_RETURN_NONE;
    if (!PyLong_CheckExact(a[10]) || !PyLong_CheckExact(a[11]) || !PyBool_Check(a[12]) || !nothing_looks_on()) Py_RETURN_NONE;
    const DdsShape s{PyLong_AsLongLong(a[10]), PyLong_AsLongLong(a[11]), a[12] == Py_True};
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const at::Tensor &x = *t[0], &data = *t[1];
    if (!is_bare(x) || !is_bare(data) || !dds_covers(x, data, s) || s.s0 % 16 || s.s1 % 16 || t[2]->scalar_type() != at::kInt ||
        t[3]->scalar_type() != at::kShort || t[4]->scalar_type() != at::kShort)
        Py_RETURN_NONE;
    const bool record = c10::GradMode::is_enabled() && (x.requires_grad() || data.requires_grad());
    for (int i = 0; i < 8; ++i)
        if (record && t[i]->is_inference()) Py_RETURN_NONE;
    PyObject *flag = s.tb ? Py_False : Py_True;
    Py_INCREF(flag);
    const PyOwned held(look_up(a[0], *t[2], *t[4], data, s.tb ? s.s1 : s.s0, s.tb ? s.s0 : s.s1, flag));
    if (!held.o) return nullptr;
    const TopologyHandle *topo = static_cast<const TopologyHandle *>(PyLong_AsVoidPtr(PyTuple_GET_ITEM(held.o, 0)));
    if (!topo || topo->Rb >= 1 << 26) Py_RETURN_NONE;
    at::Tensor y = record ? DdsFn::apply(x, data, *t[2], *t[3], *t[4], *t[5], *t[6], *t[7], s, DdsCall{topo, a[0], a[1]}) : run_dds(topo, x, data);
    return THPVariable_Wrap(std::move(y));
}

template <PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *self, PyObject *const *a, Py_ssize_t na) {      // torch's C++ exceptions (out of memory) as Python ones
    HANDLE_TH_ERRORS
    return F(self, a, na);
    END_HANDLE_TH_ERRORS
}

#define MORTAR_METHOD(name, f, doc) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(guarded<f>)), METH_FASTCALL, doc}
PyMethodDef methods[] = {
    MORTAR_METHOD("mlp", py_mlp, "The carved MLP on the rows of x, or None when the call is not covered."),
    MORTAR_METHOD("routed_decode", py_routed_decode, "RMSNorm, router and gated MLP for decode rows, or None."),
    MORTAR_METHOD("route", py_route, "The router of the rows of x and its load statistics, or None."),
    MORTAR_METHOD("gemv_f32", py_gemv_f32, "The fp32 decode product of a one-scale matrix, or None."),
    MORTAR_METHOD("train_forward", py_train_forward, "Re-pack, gate_up, SwiGLU and down of a training step, or None."),
    MORTAR_METHOD("train_backward", py_train_backward, "The gradients of a training step, or None."),
    MORTAR_METHOD("dds", py_dds, "The product over stored block values with its autograd node, or None."),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mortar_native", "Native call layer of the MORTAR runtime.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mortar_native(void) {
    const char *names[N_NAMES] = {"weight", "bias", "sub_keys_a", "sub_keys_b", "group_bias", "iter_embed"};
    for (int i = 0; i < N_NAMES; ++i)
        if (!(g_names[i] = PyUnicode_InternFromString(names[i]))) return nullptr;
    return PyModule_Create(&module);
}
