// The calls a program makes once a matrix, as methods of a C base type of jitllm_amd.device.Device.
//
// A decode matvec is about 3 us of device time, and so is the way to its launch: through Python wrappers and
// ctypes a call cost 1.5 us (a list-of-matrices call 2.5) before the C ABI was reached.  These take their
// arguments off the interpreter's stack, hand addresses straight to the ABI and cost 0.2-0.4 us.
//
// The ABI's functions are bound at run time (bind(), addresses from the loaded libjlmi.so): this module has no
// link-time dependency on the HIP runtime, so importing the package before a framework that brings its own
// runtime stays harmless.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <numpy/arrayobject.h>

#include <cstring>

#include "../../include/jlmi.h"

namespace {

struct Api {
    decltype(&jl_matvec) matvec;
    decltype(&jl_matmul) matmul;
    decltype(&jl_matvec_packed) matvec_packed;
    decltype(&jl_matmul_packed) matmul_packed;
    decltype(&jl_matvec_dev) matvec_dev;
    decltype(&jl_matvec_packed_dev) matvec_packed_dev;
    decltype(&jl_matvec_group_dev) matvec_group_dev;
    decltype(&jl_matmul_dev) matmul_dev;
    decltype(&jl_matmul_packed_dev) matmul_packed_dev;
    decltype(&jl_layer_ffn_dev) layer_ffn_dev;
    decltype(&jl_moe_block_dev) moe_block_dev;
    decltype(&jl_moe_block_packed_dev) moe_block_packed_dev;
    decltype(&jl_matmul_mxfp4_bf16_dev) matmul_mxfp4_bf16_dev;
    decltype(&jl_matmul_mxfp4_packed_bf16_dev) matmul_mxfp4_packed_bf16_dev;
} api;
PyObject *host_types, *bank_type;                                  // quant.BLOCK, _lib.PackedBank
PyObject *s_qs, *s_d, *s_sc, *s_row, *s_stride, *s_served;

struct Calls {
    PyObject_HEAD
    jl_ctx* ctx;
};

// ---- arguments
// A call's arguments in the order of `names` (the first nreq are required); absent ones stay null.
bool take(const char* fn, const char* const* names, int nreq, int nmax, PyObject* const* a, Py_ssize_t n, PyObject* kw, PyObject** out) {
    if (n > nmax) {
        PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", fn, nmax, n);
        return false;
    }
    for (int i = 0; i < nmax; i++) out[i] = i < n ? a[i] : nullptr;
    const Py_ssize_t nk = kw ? PyTuple_GET_SIZE(kw) : 0;
    for (Py_ssize_t j = 0; j < nk; j++) {
        PyObject* key = PyTuple_GET_ITEM(kw, j);
        int at = 0;
        while (at < nmax && PyUnicode_CompareWithASCIIString(key, names[at]) != 0) at++;
        if (at == nmax) {
            PyErr_Format(PyExc_TypeError, "%s() got an unexpected keyword argument '%U'", fn, key);
            return false;
        }
        if (out[at]) {
            PyErr_Format(PyExc_TypeError, "%s() got multiple values for argument '%s'", fn, names[at]);
            return false;
        }
        out[at] = a[n + j];
    }
    for (int i = 0; i < nreq; i++)
        if (!out[i]) {
            PyErr_Format(PyExc_TypeError, "%s() missing required argument: '%s'", fn, names[i]);
            return false;
        }
    return true;
}

// An address: a Python integer, a numpy array's data, or whatever int() makes of the object.
bool ptr(PyObject* o, void** p) {
    if (PyLong_Check(o)) {
        *p = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(o);
        return !PyErr_Occurred();
    }
    if (PyArray_Check(o)) {
        *p = PyArray_DATA((PyArrayObject*)o);
        return true;
    }
    PyObject* v = PyNumber_Long(o);
    if (!v) return false;
    *p = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(v);
    Py_DECREF(v);
    return !PyErr_Occurred();
}
bool opt(PyObject* o, void** p) {
    *p = nullptr;
    return !o || o == Py_None || ptr(o, p);
}
bool num(PyObject* o, int* v) {
    const long l = PyLong_AsLong(o);
    if (l == -1 && PyErr_Occurred()) return false;
    *v = (int)l;
    return true;
}
bool real(PyObject* o, float* v) {
    if (!o) return true;
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return false;
    *v = (float)d;
    return true;
}
// The stream argument: None or an address (an int, or a ctypes pointer).
bool stream_of(PyObject* o, void** p) {
    *p = nullptr;
    if (!o || o == Py_None) return true;
    if (PyLong_Check(o)) return ptr(o, p);
    PyObject* v = PyObject_GetAttrString(o, "value");
    if (!v) return false;
    const bool ok = opt(v, p);
    Py_DECREF(v);
    return ok;
}

PyObject* ended(Calls* self, int rc, const char* what) {
    if (rc == JL_OK) Py_RETURN_TRUE;
    if (rc == JL_DECLINED) Py_RETURN_FALSE;
    PyObject *c = PyLong_FromLong(rc), *w = PyUnicode_FromString(what);
    PyObject* r = c && w ? PyObject_CallMethodObjArgs((PyObject*)self, s_served, c, w, nullptr) : nullptr;   // raises DeviceError
    Py_XDECREF(c);
    Py_XDECREF(w);
    return r;
}

template <class F> int unlocked(F f) {   // the interpreter goes on meanwhile, as under ctypes
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}

bool attr_ptr(PyObject* o, PyObject* name, void** p, bool may_be_none) {
    PyObject* v = PyObject_GetAttr(o, name);
    if (!v) return false;
    const bool ok = may_be_none ? opt(v, p) : ptr(v, p);
    Py_DECREF(v);
    return ok;
}
bool attr_num(PyObject* o, PyObject* name, int* n) {
    PyObject* v = PyObject_GetAttr(o, name);
    if (!v) return false;
    const bool ok = num(v, n);
    Py_DECREF(v);
    return ok;
}
struct Planes {
    void *qs = nullptr, *d = nullptr, *sc = nullptr;
    int row = 0, stride = 0;
    bool of(PyObject* o) {
        return attr_ptr(o, s_qs, &qs, false) && attr_ptr(o, s_d, &d, false) && attr_ptr(o, s_sc, &sc, true) && attr_num(o, s_row, &row) &&
               attr_num(o, s_stride, &stride);
    }
};

#define TAKE(fn, nreq, ...)                                              \
    static const char* const names[] = {__VA_ARGS__};                    \
    constexpr int N = (int)(sizeof names / sizeof names[0]);             \
    PyObject* a[N];                                                      \
    if (!take(fn, names, nreq, N, av, an, kw, a)) return nullptr
#define SIG Calls *self, PyObject *const *av, Py_ssize_t an, PyObject *kw

// ---- device pointers
PyObject* py_matvec_dev(SIG) {
    TAKE("matvec_dev", 6, "out", "t", "w", "x", "nrows", "k", "stream");
    void *out, *w, *x, *st;
    int t, nrows, k;
    if (!ptr(a[0], &out) || !num(a[1], &t) || !ptr(a[2], &w) || !ptr(a[3], &x) || !num(a[4], &nrows) || !num(a[5], &k) || !stream_of(a[6], &st)) return nullptr;
    return ended(self, unlocked([&] { return api.matvec_dev(self->ctx, (float*)out, t, w, (const float*)x, nrows, k, st); }), "jl_matvec_dev");
}

PyObject* py_matvec_packed_dev(SIG) {
    TAKE("matvec_packed_dev", 6, "out", "t", "p", "x", "nrows", "k", "stream");
    void *out, *x, *st;
    int t, nrows, k;
    Planes p;
    if (!ptr(a[0], &out) || !num(a[1], &t) || !p.of(a[2]) || !ptr(a[3], &x) || !num(a[4], &nrows) || !num(a[5], &k) || !stream_of(a[6], &st)) return nullptr;
    return ended(self, unlocked([&] {
        return api.matvec_packed_dev(self->ctx, (float*)out, t, (uint32_t*)p.qs, (uint32_t*)p.d, (uint32_t*)p.sc, p.row, p.stride, (const float*)x, nrows, k, st);
    }), "jl_matvec_packed_dev");
}

PyObject* py_matmul_dev(SIG) {
    TAKE("matmul_dev", 7, "out", "t", "w", "x", "nrows", "k", "ntok", "stream");
    void *out, *w, *x, *st;
    int t, nrows, k, ntok;
    if (!ptr(a[0], &out) || !num(a[1], &t) || !ptr(a[2], &w) || !ptr(a[3], &x) || !num(a[4], &nrows) || !num(a[5], &k) || !num(a[6], &ntok) || !stream_of(a[7], &st)) return nullptr;
    return ended(self, unlocked([&] { return api.matmul_dev(self->ctx, (float*)out, t, w, (const float*)x, nrows, k, ntok, st); }), "jl_matmul_dev");
}

PyObject* py_matmul_packed_dev(SIG) {
    TAKE("matmul_packed_dev", 7, "out", "t", "p", "x", "nrows", "k", "ntok", "stream");
    void *out, *x, *st;
    int t, nrows, k, ntok;
    Planes p;
    if (!ptr(a[0], &out) || !num(a[1], &t) || !p.of(a[2]) || !ptr(a[3], &x) || !num(a[4], &nrows) || !num(a[5], &k) || !num(a[6], &ntok) || !stream_of(a[7], &st)) return nullptr;
    return ended(self, unlocked([&] {
        return api.matmul_packed_dev(self->ctx, (float*)out, t, (uint32_t*)p.qs, (uint32_t*)p.d, (uint32_t*)p.sc, p.row, p.stride, (const float*)x, nrows, k, ntok, st);
    }), "jl_matmul_packed_dev");
}

PyObject* py_matmul_mxfp4_bf16_dev(SIG) {
    TAKE("matmul_mxfp4_bf16_dev", 6, "out", "w", "x", "nrows", "k", "ntok", "stream");
    void *out, *w, *x, *st;
    int nrows, k, ntok;
    if (!ptr(a[0], &out) || !ptr(a[1], &w) || !ptr(a[2], &x) || !num(a[3], &nrows) || !num(a[4], &k) || !num(a[5], &ntok) || !stream_of(a[6], &st)) return nullptr;
    return ended(self, unlocked([&] { return api.matmul_mxfp4_bf16_dev(self->ctx, (float*)out, w, (const uint16_t*)x, nrows, k, ntok, st); }), "jl_matmul_mxfp4_bf16_dev");
}

PyObject* py_matmul_mxfp4_packed_bf16_dev(SIG) {
    TAKE("matmul_mxfp4_packed_bf16_dev", 6, "out", "p", "x", "nrows", "k", "ntok", "stream");
    void *out, *x, *st;
    int nrows, k, ntok;
    Planes p;
    if (!ptr(a[0], &out) || !p.of(a[1]) || !ptr(a[2], &x) || !num(a[3], &nrows) || !num(a[4], &k) || !num(a[5], &ntok) || !stream_of(a[6], &st)) return nullptr;
    return ended(self, unlocked([&] {
        return api.matmul_mxfp4_packed_bf16_dev(self->ctx, (float*)out, (uint32_t*)p.qs, (uint32_t*)p.d, p.row, p.stride, (const uint16_t*)x, nrows, k, ntok, st);
    }), "jl_matmul_mxfp4_packed_bf16_dev");
}

PyObject* py_layer_ffn_dev(SIG) {
    TAKE("layer_ffn_dev", 4, "li", "h", "resid", "n", "stream");
    void *h, *resid, *st;
    int li, n;
    if (!num(a[0], &li) || !ptr(a[1], &h) || !ptr(a[2], &resid) || !num(a[3], &n) || !stream_of(a[4], &st)) return nullptr;
    return ended(self, unlocked([&] { return api.layer_ffn_dev(self->ctx, li, (const float*)h, (float*)resid, n, st); }), "jl_layer_ffn_dev");
}

// Up to JL_MAX_GROUP items of a sequence through `f`, which gets (index, item).
template <class F> bool each(PyObject* seq, int n, F f) {
    PyObject* s = PySequence_Fast(seq, "a sequence of a group's matrices");
    if (!s) return false;
    bool ok = PySequence_Fast_GET_SIZE(s) >= n;
    if (!ok) PyErr_SetString(PyExc_IndexError, "a group's sequences differ in length");
    for (int i = 0; i < n && ok; i++) ok = f(i, PySequence_Fast_GET_ITEM(s, i));
    Py_DECREF(s);
    return ok;
}

PyObject* py_matvec_group_dev(SIG) {
    TAKE("matvec_group_dev", 6, "outs", "types", "ws", "rows", "x", "k", "act_up", "resid", "alpha", "stream", "norm_w", "norm_eps", "norm_out", "resid_gate");
    const Py_ssize_t n = PySequence_Size(a[0]);
    if (n < 0) return nullptr;
    if (n > JL_MAX_GROUP) {
        PyErr_Format(PyExc_IndexError, "a group holds up to %d matrices", JL_MAX_GROUP);
        return nullptr;
    }
    jl_mv_group g;
    memset(&g, 0, sizeof g);
    g.n = (int)n;
    void *x, *up, *resid, *nw, *no, *rg, *st, *p;
    if (!each(a[0], g.n, [&](int i, PyObject* o) { return ptr(o, &p) && (g.out[i] = (float*)p, true); }) ||
        !each(a[1], g.n, [&](int i, PyObject* o) { return num(o, &g.type[i]); }) ||
        !each(a[2], g.n, [&](int i, PyObject* o) { return ptr(o, &p) && (g.w[i] = p, true); }) ||
        !each(a[3], g.n, [&](int i, PyObject* o) { return num(o, &g.rows[i]); }) || !ptr(a[4], &x) || !num(a[5], &g.k) || !opt(a[6], &up) ||
        !opt(a[7], &resid) || !real(a[8], &g.alpha) || !stream_of(a[9], &st) || !opt(a[10], &nw) || !real(a[11], &g.norm_eps) ||
        !opt(a[12], &no) || !opt(a[13], &rg))
        return nullptr;
    g.x = (const float*)x; g.act_up = (const float*)up; g.resid = (float*)resid;
    g.norm_w = (const float*)nw; g.norm_out = (float*)no; g.resid_gate = (const float*)rg;
    return ended(self, unlocked([&] { return api.matvec_group_dev(self->ctx, &g, st); }), "jl_matvec_group_dev");
}

PyObject* py_moe_block_dev(SIG) {
    TAKE("moe_block_dev", 12, "resid", "t", "gate", "up", "down", "router", "x", "rows", "k_used", "n_expert", "n_ffn", "n_embd", "sel", "wt", "stream",
         "down_type", "router_type");
    void *resid, *router, *x, *sel, *wt, *st;
    int t, rows, k_used, ne, n_ffn, n_embd, dt, rt = 0;
    if (!ptr(a[0], &resid) || !num(a[1], &t) || !ptr(a[5], &router) || !ptr(a[6], &x) || !num(a[7], &rows) || !num(a[8], &k_used) ||
        !num(a[9], &ne) || !num(a[10], &n_ffn) || !num(a[11], &n_embd) || !opt(a[12], &sel) || !opt(a[13], &wt) || !stream_of(a[14], &st) ||
        (a[16] && !num(a[16], &rt)))
        return nullptr;
    const int packed = PyObject_IsInstance(a[2], bank_type);
    if (packed < 0) return nullptr;
    if (packed) {
        Py_buffer b[3];
        int got = 0;
        for (; got < 3; got++) {
            const int is = PyObject_IsInstance(a[2 + got], bank_type);
            if (is <= 0 || PyObject_GetBuffer(a[2 + got], &b[got], PyBUF_SIMPLE) != 0) {
                if (is == 0) PyErr_SetString(PyExc_TypeError, "moe_block_dev(): gate, up and down are three packed banks or three addresses");
                break;
            }
        }
        PyObject* r = nullptr;
        if (got == 3) {
            const jl_packed_bank *g = (const jl_packed_bank*)b[0].buf, *u = (const jl_packed_bank*)b[1].buf, *d = (const jl_packed_bank*)b[2].buf;
            r = ended(self, unlocked([&] {
                return api.moe_block_packed_dev(self->ctx, (float*)resid, t, g, u, d, rt, router, (const float*)x, rows, k_used, ne, n_ffn, n_embd, (uint32_t*)sel, (float*)wt, st);
            }), "jl_moe_block_packed_dev");
        }
        for (int i = 0; i < got; i++) PyBuffer_Release(&b[i]);
        return r;
    }
    void *g, *u, *d;
    dt = t;
    if (!ptr(a[2], &g) || !ptr(a[3], &u) || !ptr(a[4], &d) || (a[15] && a[15] != Py_None && !num(a[15], &dt))) return nullptr;
    return ended(self, unlocked([&] {
        return api.moe_block_dev(self->ctx, (float*)resid, t, dt, g, u, d, rt, router, (const float*)x, rows, k_used, ne, n_ffn, n_embd, (uint32_t*)sel, (float*)wt, st);
    }), "jl_moe_block_dev");
}

// ---- host memory: numpy arrays, checked
bool is(PyObject* o, int type) {
    return PyArray_Check(o) && PyArray_TYPE((PyArrayObject*)o) == type && PyArray_ISNOTSWAPPED((PyArrayObject*)o);
}
bool hold(bool ok, const char* what) {
    if (!ok) PyErr_SetString(PyExc_AssertionError, what);
    return ok;
}
#define DATA(o) PyArray_DATA((PyArrayObject*)(o))

PyObject* host_rows(Calls* self, PyObject** a, int ntok, const char* what) {
    const int known = PySequence_Contains(host_types, a[1]);
    if (known < 0) return nullptr;
    if (!known) Py_RETURN_FALSE;
    int t, nrows, k;
    if (!hold(is(a[0], NPY_FLOAT32) && is(a[3], NPY_FLOAT32) && is(a[2], NPY_UINT8), "out and x are float32 arrays, w a uint8 array") || !num(a[1], &t) ||
        !num(a[4], &nrows) || !num(a[5], &k))
        return nullptr;
    if (!hold(PyArray_SIZE((PyArrayObject*)a[0]) >= (npy_intp)ntok * nrows && PyArray_SIZE((PyArrayObject*)a[3]) >= (npy_intp)ntok * k, "out or x is too small"))
        return nullptr;
    float *out = (float*)DATA(a[0]), *x = (float*)DATA(a[3]);
    void* w = DATA(a[2]);
    const size_t wb = (size_t)PyArray_NBYTES((PyArrayObject*)a[2]);
    return ended(self, unlocked([&] { return api.matmul(self->ctx, out, t, w, wb, x, nrows, k, ntok); }), what);
}
PyObject* py_MatVec(SIG) {
    TAKE("MatVec", 6, "out", "t", "w", "x", "nrows", "k");
    return host_rows(self, a, 1, "jl_matvec");
}
PyObject* py_MatMul(SIG) {
    TAKE("MatMul", 7, "out", "t", "w", "x", "nrows", "k", "ntok");
    int ntok;
    if (!num(a[6], &ntok)) return nullptr;
    return host_rows(self, a, ntok, "jl_matmul");
}

PyObject* host_planes(Calls* self, PyObject** a, int ntok, const char* what) {
    int t, nrows, k;
    Planes p;
    if (!hold(is(a[0], NPY_FLOAT32) && is(a[3], NPY_FLOAT32), "out and x are float32 arrays") || !num(a[1], &t) || !p.of(a[2]) || !num(a[4], &nrows) || !num(a[5], &k))
        return nullptr;
    float *out = (float*)DATA(a[0]), *x = (float*)DATA(a[3]);
    return ended(self, unlocked([&] {
        return api.matmul_packed(self->ctx, out, t, (uint32_t*)p.qs, (uint32_t*)p.d, (uint32_t*)p.sc, p.row, p.stride, x, nrows, k, ntok);
    }), what);
}
PyObject* py_MatVecPacked(SIG) {
    TAKE("MatVecPacked", 6, "out", "t", "p", "x", "nrows", "k");
    return host_planes(self, a, 1, "jl_matvec_packed");
}
PyObject* py_MatMulPacked(SIG) {
    TAKE("MatMulPacked", 7, "out", "t", "p", "x", "nrows", "k", "ntok");
    int ntok;
    if (!num(a[6], &ntok)) return nullptr;
    return host_planes(self, a, ntok, "jl_matmul_packed");
}

PyObject* py_attach(Calls* self, PyObject* ctx) {   // _attach(address): the context the calls go to; None: none
    void* p;
    if (!opt(ctx, &p)) return nullptr;
    self->ctx = (jl_ctx*)p;
    Py_RETURN_NONE;
}

#define M(name, doc) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL | METH_KEYWORDS, doc}
PyMethodDef methods[] = {
    {"_attach", (PyCFunction)py_attach, METH_O, nullptr},
    M(matvec_dev, "matvec_dev(out, t, w, x, nrows, k, stream=None): out[0:nrows] = W x on device operands."),
    M(matvec_packed_dev, "matvec_packed_dev(out, t, p, x, nrows, k, stream=None): the same over packed planes; p = Packed(...)."),
    M(matvec_group_dev,
      "matvec_group_dev(outs, types, ws, rows, x, k, act_up=None, resid=None, alpha=0.0, stream=None, norm_w=None, norm_eps=0.0,\n"
      "norm_out=None, resid_gate=None).  JIT.MatVecPackedGroup: up to four matvecs reading one activation, optional\n"
      "RMSNorm(x) * norm_w first, optional silu(x) * act_up and resid += alpha * out[0]\n"
      "(alpha * sigmoid(*resid_gate) when a device logit gates the add), in one launch."),
    M(matmul_dev, "matmul_dev(out, t, w, x, nrows, k, ntok, stream=None): x [ntok][k] -> out [ntok][nrows] on device operands\n"
                  "(JIT.MatMulPacked semantics)."),
    M(matmul_packed_dev, "matmul_packed_dev(out, t, p, x, nrows, k, ntok, stream=None): the same over packed planes."),
    M(matmul_mxfp4_bf16_dev, "matmul_mxfp4_bf16_dev(out, w, x, nrows, k, ntok, stream=None): MXFP4 weights x bf16 activations (bits as\n"
                             "uint16) -> f32 out [ntok][nrows]."),
    M(matmul_mxfp4_packed_bf16_dev, "matmul_mxfp4_packed_bf16_dev(out, p, x, nrows, k, ntok, stream=None): the same over packed MXFP4 planes;\n"
                                    "p = Packed(qs, d, None, row, stride)."),
    M(layer_ffn_dev, "layer_ffn_dev(li, h, resid, n, stream=None): run prepared block li's feed-forward for n rows:\n"
                     "resid [n][n_embd] += ffn(h [n][n_embd])."),
    M(moe_block_dev,
      "moe_block_dev(resid, t, gate, up, down, router, x, rows, k_used, n_expert, n_ffn, n_embd, sel=None, wt=None, stream=None,\n"
      "down_type=None, router_type=0).  The whole mixture block, router included: resid [rows][n_embd] += mixture output.\n"
      "gate / up / down: banks of GGUF sheets (device addresses), or three packed_bank(...) structures."),
    M(MatVec, "MatVec(out, t, w, x, nrows, k).  nn.Device.MatVec: out[0:nrows] = W x over raw GGUF bytes; False = declined."),
    M(MatMul, "MatMul(out, t, w, x, nrows, k, ntok).  JIT.MatMul (/root/reference/engine/nn/matmul.go:27): x [ntok][k] -> out [ntok][nrows]."),
    M(MatVecPacked, "MatVecPacked(out, t, p, x, nrows, k).  JIT.MatVecPacked (/root/reference/engine/nn/packed.go:24);\n"
                    "p = Packed(qs, d, sc, row, stride)."),
    M(MatMulPacked, "MatMulPacked(out, t, p, x, nrows, k, ntok).  JIT.MatMulPacked (/root/reference/engine/nn/packedmm.go:23)."),
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject calls_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// bind(addresses by name of the C ABI, the block types host calls serve, the packed bank structure)
PyObject* py_bind(PyObject*, PyObject* args) {
    PyObject *fns, *types, *bank;
    if (!PyArg_ParseTuple(args, "O!OO", &PyDict_Type, &fns, &types, &bank)) return nullptr;
#define FN(field)                                                                     \
    {                                                                                 \
        PyObject* o = PyDict_GetItemString(fns, "jl_" #field);                        \
        void* p;                                                                      \
        if (!o) return PyErr_Format(PyExc_KeyError, "bind: no address of jl_" #field); \
        if (!ptr(o, &p)) return nullptr;                                              \
        api.field = (decltype(api.field))p;                                           \
    }
    FN(matvec) FN(matmul) FN(matvec_packed) FN(matmul_packed) FN(matvec_dev) FN(matvec_packed_dev) FN(matvec_group_dev) FN(matmul_dev)
    FN(matmul_packed_dev) FN(layer_ffn_dev) FN(moe_block_dev) FN(moe_block_packed_dev) FN(matmul_mxfp4_bf16_dev) FN(matmul_mxfp4_packed_bf16_dev)
#undef FN
    Py_INCREF(types);
    Py_INCREF(bank);
    Py_XSETREF(host_types, types);
    Py_XSETREF(bank_type, bank);
    Py_RETURN_NONE;
}

PyMethodDef functions[] = {{"bind", py_bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "The hot calls of jitllm_amd.device.Device.", -1, functions, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
    import_array();
    calls_type.tp_name = "jitllm_amd._calls.Calls";
    calls_type.tp_basicsize = sizeof(Calls);
    calls_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    calls_type.tp_methods = methods;
    calls_type.tp_new = PyType_GenericNew;
    if (PyType_Ready(&calls_type) < 0) return nullptr;
    s_qs = PyUnicode_InternFromString("qs"); s_d = PyUnicode_InternFromString("d"); s_sc = PyUnicode_InternFromString("sc");
    s_row = PyUnicode_InternFromString("row"); s_stride = PyUnicode_InternFromString("stride"); s_served = PyUnicode_InternFromString("_served");
    if (!s_qs || !s_d || !s_sc || !s_row || !s_stride || !s_served) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&calls_type);
    if (PyModule_AddObject(m, "Calls", (PyObject*)&calls_type) < 0) return nullptr;
    return m;
}
