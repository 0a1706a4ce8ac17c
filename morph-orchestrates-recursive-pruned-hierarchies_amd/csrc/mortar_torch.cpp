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
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mortar_hip.h"

namespace {

// One packed matrix as the Python side hands it over (pack.MortarPack.handle): the struct of the C-ABI and the two
// schedules, null until the Python side has built them.
struct PackHandle {
    const mortar_bcsr_t *w;
    const int32_t *sched1, *sched2;
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
    if (n.on && !(gu->w->seg_cb >= gu->w->Cb && mortar_norm_fusable(gu->w->Cb))) {
        xn = new_bf16(x, {M, d});
        const int rc = mortar_rmsnorm_bf16(xp, M, (int32_t)d, d, n.w, n.eps, u16m(xn), d, st);
        if (rc) return rc;
        xp = u16(xn);
        n = Norm{};
    }
    if (M > DECODE_MAX_ROWS) {
        const at::Tensor h = at::empty({mortar_mlp_hidden_bytes(M, (int32_t)f)}, x.options().dtype(at::kByte).requires_grad(false));
        return mortar_mlp_bf16(gu->w, gu->sched2, dn->w, dn->sched1, xp, M, d, n.on, n.w, n.eps, gates, ncl, h.data_ptr(), y, dy, 0, st);
    }
    const at::Tensor h = new_bf16(x, {M, f});
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
    int rc = mortar_rmsnorm_bf16(u16(x), M, (int32_t)d, d, nm.w, nm.eps, u16m(xn), d, st);
    if (rc == MORTAR_OK)
        rc = mortar_router_bf16(u16(xn), 0, M, (int32_t)d, d, r.wq, r.iter_vec, r.ln_w, r.ln_b, (float)ln_eps, r.ka, r.kb, r.nsk, r.bias,
                                r.n, (int32_t)sh[3], qv, nullptr, gates, nullptr, st);
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
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mortar_native", "Native call layer of the MORTAR runtime.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mortar_native(void) {
    const char *names[N_NAMES] = {"weight", "bias", "sub_keys_a", "sub_keys_b", "group_bias", "iter_embed"};
    for (int i = 0; i < N_NAMES; ++i)
        if (!(g_names[i] = PyUnicode_InternFromString(names[i]))) return nullptr;
    return PyModule_Create(&module);
}
