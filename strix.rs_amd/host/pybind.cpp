// The hot calls of the C ABI as a CPython extension module (_smx_native).  A decode step is launches of a few microseconds,
// and what a ctypes call spends around one of them is of that order: converting a numpy argument to a pointer through
// ndarray.ctypes costs 1.4 us, three conversions and the key's encode() 2.6 us of the 18 us of a host-pointer gemv.  Here a
// numpy array is read through the buffer protocol (0.1 us) and a key through the string's cached UTF-8 form.
//
// Every function takes the context's address first and returns the C ABI's code; the wrapper class turns that into True /
// False / SmxError.  A host array that is not C-contiguous with the expected element type makes the function return None
// (nothing has run): the wrapper converts it and calls again.  The interpreter lock is released around every call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>

#include "../../include/strix_mi355.h"

namespace {

constexpr Py_ssize_t kMaxGroup = 64;   // items of a batch converted on the stack

bool to_ptr(PyObject* o, void** p) {   // an address as int, None, or an object with .value (ctypes.c_void_p)
    if (o == Py_None) {
        *p = nullptr;
        return true;
    }
    if (PyLong_Check(o)) {
        *p = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(o);
        return !PyErr_Occurred();
    }
    PyObject* v = PyObject_GetAttrString(o, "value");
    if (!v) return false;
    const bool ok = (v == Py_None || PyLong_Check(v)) && to_ptr(v, p);
    if (!ok && !PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "an address is an int, None or a c_void_p");
    Py_DECREF(v);
    return ok;
}
template <class T>
bool to_ptr(PyObject* o, T** p) {
    void* v = nullptr;
    if (!to_ptr(o, &v)) return false;
    *p = (T*)v;
    return true;
}
bool to_size(PyObject* o, size_t* n) {
    PyObject* i = PyNumber_Index(o);
    if (!i) return false;
    *n = (size_t)PyLong_AsUnsignedLongLongMask(i);
    Py_DECREF(i);
    return !PyErr_Occurred();
}
bool to_int(PyObject* o, int* n) {
    PyObject* i = PyNumber_Index(o);
    if (!i) return false;
    *n = (int)PyLong_AsLong(i);
    Py_DECREF(i);
    return !PyErr_Occurred();
}
bool to_float(PyObject* o, float* f) {
    *f = (float)PyFloat_AsDouble(o);
    return !PyErr_Occurred();
}
bool to_key(PyObject* o, const char** k) {
    *k = PyUnicode_AsUTF8(o);
    return *k != nullptr;
}
bool argc_is(Py_ssize_t n, Py_ssize_t want) {
    if (n == want) return true;
    PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", want, n);
    return false;
}

// A C-contiguous array of `size`-byte elements whose format character is one of `kinds`.
struct Array {
    Py_buffer b;
    bool held = false;
    // 1: held; 0: another layout or element type (no exception set)
    bool get(PyObject* o, const char* kinds, Py_ssize_t size, bool writable = false) {
        if (PyObject_GetBuffer(o, &b, PyBUF_FORMAT | PyBUF_C_CONTIGUOUS | (writable ? PyBUF_WRITABLE : 0)) != 0) {
            PyErr_Clear();
            return false;
        }
        held = true;
        if (b.itemsize != size || !b.format || b.format[1] != '\0') return false;
        for (const char* k = kinds; *k; k++)
            if (b.format[0] == *k) return true;
        return false;
    }
    size_t count() const { return (size_t)(b.len / b.itemsize); }
    ~Array() {
        if (held) PyBuffer_Release(&b);
    }
};

#define ALLOW(expr)                              \
    int rc;                                      \
    Py_BEGIN_ALLOW_THREADS rc = (expr);          \
    Py_END_ALLOW_THREADS return PyLong_FromLong(rc)

#define FN(name) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)

// (ctx, key, xs_dev, m, y_dev)
template <int (*F)(smx_ctx*, const char*, const float*, size_t, float*)>
FN(rows_dev) {
    smx_ctx* c; const char* key; const float* x; size_t m; float* y;
    if (!argc_is(n, 5) || !to_ptr(a[0], &c) || !to_key(a[1], &key) || !to_ptr(a[2], &x) || !to_size(a[3], &m) || !to_ptr(a[4], &y)) return nullptr;
    ALLOW(F(c, key, x, m, y));
}
// (ctx, key, x_dev, y_dev)
FN(gemv_f32_dev) {
    smx_ctx* c; const char* key; const float* x; float* y;
    if (!argc_is(n, 4) || !to_ptr(a[0], &c) || !to_key(a[1], &key) || !to_ptr(a[2], &x) || !to_ptr(a[3], &y)) return nullptr;
    ALLOW(smx_gemv_f32_dev(c, key, x, y));
}
// (ctx, key, act, a_dev, b_dev, m, eps, y_dev)
FN(gemm_fused_dev) {
    smx_ctx* c; const char* key; int act; const float *x, *b; size_t m; float eps; float* y;
    if (!argc_is(n, 8) || !to_ptr(a[0], &c) || !to_key(a[1], &key) || !to_int(a[2], &act) || !to_ptr(a[3], &x) || !to_ptr(a[4], &b) ||
        !to_size(a[5], &m) || !to_float(a[6], &eps) || !to_ptr(a[7], &y)) return nullptr;
    ALLOW(smx_gemm_fused_dev(c, key, act, x, b, m, eps, y));
}
// (ctx, gate_key, up_key, act, x_dev, norm, norm_w_dev, eps, h_dev)
FN(ffn_gate_up_dev) {
    smx_ctx* c; const char *g, *u; int act, norm; const float *x, *w; float eps; float* h;
    if (!argc_is(n, 9) || !to_ptr(a[0], &c) || !to_key(a[1], &g) || !to_key(a[2], &u) || !to_int(a[3], &act) || !to_ptr(a[4], &x) ||
        !to_int(a[5], &norm) || !to_ptr(a[6], &w) || !to_float(a[7], &eps) || !to_ptr(a[8], &h)) return nullptr;
    ALLOW(smx_ffn_gate_up_dev(c, g, u, act, x, norm, w, eps, h));
}
// A caller's sequence, its items held until the call has returned: the library reads the keys with the interpreter lock
// released, when nothing else need keep them alive (a sequence that makes its items when asked, as a numpy array of strings
// does; a list that another thread changes).
struct Items {
    PyObject* t = nullptr;
    bool take(PyObject* iterable) {
        t = PySequence_Tuple(iterable);
        return t != nullptr;
    }
    Py_ssize_t count() const { return PyTuple_GET_SIZE(t); }
    PyObject* operator[](Py_ssize_t i) const { return PyTuple_GET_ITEM(t, i); }
    Items() = default;
    Items(const Items&) = delete;
    Items& operator=(const Items&) = delete;
    ~Items() { Py_XDECREF(t); }
};
// keys (anything of known length) / addresses of a group (up to the ABI's limit; more are counted and refused there)
bool to_keys(PyObject* seq, Items* held, const char** out, Py_ssize_t* count) {
    if (PyObject_Size(seq) < 0 || !held->take(seq)) return false;
    *count = held->count();
    for (Py_ssize_t i = 0; i < *count && i < kMaxGroup; i++)
        if (!to_key((*held)[i], &out[i])) return false;
    return true;
}
template <class T>
bool to_ptrs(PyObject* seq, T** out, Py_ssize_t want) {
    Items f;
    if (!f.take(seq)) return false;
    if (f.count() != want) {
        PyErr_SetString(PyExc_ValueError, "one address per key");
        return false;
    }
    for (Py_ssize_t i = 0; i < want && i < kMaxGroup; i++)
        if (!to_ptr(f[i], &out[i])) return false;
    return true;
}
// (ctx, keys, xs_dev, ys_dev)
FN(gemv_batch_dev) {
    smx_ctx* c; const char* keys[kMaxGroup] = {}; const float* xs[kMaxGroup] = {}; float* ys[kMaxGroup] = {}; Py_ssize_t k;
    Items held;
    if (!argc_is(n, 4) || !to_ptr(a[0], &c) || !to_keys(a[1], &held, keys, &k) || !to_ptrs(a[2], xs, k) || !to_ptrs(a[3], ys, k)) return nullptr;
    ALLOW(smx_gemv_batch_dev(c, (size_t)k, keys, xs, ys));
}
// (ctx, keys, act, a_dev, b_dev, eps, ys_dev)
FN(gemv_fused_dev) {
    smx_ctx* c; const char* keys[kMaxGroup] = {}; int act; const float *x, *b; float eps; float* ys[kMaxGroup] = {}; Py_ssize_t k;
    Items held;
    if (!argc_is(n, 7) || !to_ptr(a[0], &c) || !to_keys(a[1], &held, keys, &k) || !to_int(a[2], &act) || !to_ptr(a[3], &x) || !to_ptr(a[4], &b) ||
        !to_float(a[5], &eps) || !to_ptrs(a[6], ys, k)) return nullptr;
    ALLOW(smx_gemv_fused_dev(c, (size_t)k, keys, act, x, b, eps, ys));
}
// (ctx, logits_dev, ne, k, ids_dev, w_dev)
FN(moe_route_dev) {
    smx_ctx* c; const float* l; size_t ne, k; int32_t* ids; float* w;
    if (!argc_is(n, 6) || !to_ptr(a[0], &c) || !to_ptr(a[1], &l) || !to_size(a[2], &ne) || !to_size(a[3], &k) || !to_ptr(a[4], &ids) || !to_ptr(a[5], &w))
        return nullptr;
    ALLOW(smx_moe_route_dev(c, l, ne, k, ids, w));
}
// (ctx, layer, logits_dev, k, x_dev, y_dev, ids_dev, w_dev)
FN(moe_ffn_logits_dev) {
    smx_ctx* c; size_t layer, k; const float *l, *x; float *y, *w; int32_t* ids;
    if (!argc_is(n, 8) || !to_ptr(a[0], &c) || !to_size(a[1], &layer) || !to_ptr(a[2], &l) || !to_size(a[3], &k) || !to_ptr(a[4], &x) ||
        !to_ptr(a[5], &y) || !to_ptr(a[6], &ids) || !to_ptr(a[7], &w)) return nullptr;
    ALLOW(smx_moe_ffn_logits_dev(c, layer, l, k, x, y, ids, w));
}
// (ctx, layer, ids_dev, w_dev, k, x_dev, y_dev)
FN(moe_ffn_routed_dev) {
    smx_ctx* c; size_t layer, k; const int32_t* ids; const float *w, *x; float* y;
    if (!argc_is(n, 7) || !to_ptr(a[0], &c) || !to_size(a[1], &layer) || !to_ptr(a[2], &ids) || !to_ptr(a[3], &w) || !to_size(a[4], &k) ||
        !to_ptr(a[5], &x) || !to_ptr(a[6], &y)) return nullptr;
    ALLOW(smx_moe_ffn_routed_dev(c, layer, ids, w, k, x, y));
}
// (ctx, graph)
FN(graph_launch) {
    smx_ctx* c; smx_graph* g;
    if (!argc_is(n, 2) || !to_ptr(a[0], &c) || !to_ptr(a[1], &g)) return nullptr;
    ALLOW(smx_graph_launch(c, g));
}

// host arrays: (ctx, key, x, y), one row
template <int (*F)(smx_ctx*, const char*, const float*, size_t, float*, size_t)>
FN(gemv_host) {
    smx_ctx* c; const char* key; Array x, y;
    if (!argc_is(n, 4) || !to_ptr(a[0], &c) || !to_key(a[1], &key)) return nullptr;
    if (!x.get(a[2], "f", 4) || !y.get(a[3], "f", 4, true)) Py_RETURN_NONE;
    ALLOW(F(c, key, (const float*)x.b.buf, x.count(), (float*)y.b.buf, y.count()));
}
// (ctx, key, xs, m, y): m rows
template <int (*F)(smx_ctx*, const char*, const float*, size_t, size_t, float*, size_t)>
FN(rows_host) {
    smx_ctx* c; const char* key; Array x, y; size_t m;
    if (!argc_is(n, 5) || !to_ptr(a[0], &c) || !to_key(a[1], &key) || !to_size(a[3], &m)) return nullptr;
    if (!x.get(a[2], "f", 4) || !y.get(a[4], "f", 4, true) || m == 0 || x.count() % m != 0) Py_RETURN_NONE;
    ALLOW(F(c, key, (const float*)x.b.buf, m, x.count() / m, (float*)y.b.buf, y.count()));
}
// (ctx, key, xs, m, out u32[m])
FN(lm_head_argmax_rows) {
    smx_ctx* c; const char* key; Array x, y; size_t m;
    if (!argc_is(n, 5) || !to_ptr(a[0], &c) || !to_key(a[1], &key) || !to_size(a[3], &m)) return nullptr;
    if (!x.get(a[2], "f", 4) || !y.get(a[4], "I", 4, true) || m == 0 || x.count() % m != 0 || y.count() < m) Py_RETURN_NONE;
    ALLOW(smx_lm_head_argmax_rows(c, key, (const float*)x.b.buf, m, x.count() / m, (uint32_t*)y.b.buf));
}
// (ctx, f32, calls [(key, x)], ys): the ABI's code, or the items' codes as a list when one of them is not 1
FN(gemv_batch) {
    smx_ctx* c; int f32;
    if (!argc_is(n, 4) || !to_ptr(a[0], &c) || !to_int(a[1], &f32)) return nullptr;
    if (!PyList_Check(a[2]) || !PyList_Check(a[3])) Py_RETURN_NONE;
    Items calls, outs;
    if (!calls.take(a[2]) || !outs.take(a[3])) return nullptr;
    const Py_ssize_t k = calls.count();
    if (k > kMaxGroup || outs.count() != k) Py_RETURN_NONE;
    const char* keys[kMaxGroup]; const float* xs[kMaxGroup]; float* ys[kMaxGroup]; size_t il[kMaxGroup], oc[kMaxGroup]; int st[kMaxGroup];
    Array x[kMaxGroup], y[kMaxGroup];
    for (Py_ssize_t i = 0; i < k; i++) {
        PyObject* t = calls[i];
        if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != 2) Py_RETURN_NONE;
        if (!to_key(PyTuple_GET_ITEM(t, 0), &keys[i])) return nullptr;
        if (!x[i].get(PyTuple_GET_ITEM(t, 1), "f", 4) || !y[i].get(outs[i], "f", 4, true)) Py_RETURN_NONE;
        xs[i] = (const float*)x[i].b.buf; il[i] = x[i].count();
        ys[i] = (float*)y[i].b.buf; oc[i] = y[i].count();
        st[i] = 0;
    }
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = f32 ? smx_gemv_f32_batch(c, (size_t)k, keys, xs, il, ys, oc, st) : smx_gemv_batch(c, (size_t)k, keys, xs, il, ys, oc, st);
    Py_END_ALLOW_THREADS
    bool all = rc == SMX_OK;
    for (Py_ssize_t i = 0; all && i < k; i++) all = st[i] == SMX_OK;
    if (all || rc != SMX_OK) return PyLong_FromLong(rc);
    PyObject* l = PyList_New(k);
    for (Py_ssize_t i = 0; l && i < k; i++) PyList_SET_ITEM(l, i, PyLong_FromLong(st[i]));
    return l;
}
// (ctx, layer, ids i32, wexp, x, sgate, y)
FN(moe_ffn) {
    smx_ctx* c; size_t layer; Array ids, w, x, y; float sgate;
    if (!argc_is(n, 7) || !to_ptr(a[0], &c) || !to_size(a[1], &layer) || !to_float(a[5], &sgate)) return nullptr;
    if (!ids.get(a[2], "i", 4) || !w.get(a[3], "f", 4) || !x.get(a[4], "f", 4) || !y.get(a[6], "f", 4, true) || w.count() < ids.count()) Py_RETURN_NONE;
    ALLOW(smx_moe_ffn(c, layer, (const int32_t*)ids.b.buf, (const float*)w.b.buf, ids.count(), (const float*)x.b.buf, x.count(), sgate,
                      (float*)y.b.buf, y.count()));
}
// (ctx, layer, ids i32, wexp, x_dev, y_dev)
FN(moe_ffn_dev) {
    smx_ctx* c; size_t layer; Array ids, w; const float* x; float* y;
    if (!argc_is(n, 6) || !to_ptr(a[0], &c) || !to_size(a[1], &layer) || !to_ptr(a[4], &x) || !to_ptr(a[5], &y)) return nullptr;
    if (!ids.get(a[2], "i", 4) || !w.get(a[3], "f", 4) || w.count() < ids.count()) Py_RETURN_NONE;
    ALLOW(smx_moe_ffn_dev(c, layer, (const int32_t*)ids.b.buf, (const float*)w.b.buf, ids.count(), x, y));
}
// (ctx, layer, xs_dev, m, plan [nplan][3] 64-bit, slot_tok i32, wslot, y_dev)
FN(moe_layer_dev) {
    smx_ctx* c; size_t layer, m; const float* x; float* y; Array plan, tok, w;
    if (!argc_is(n, 8) || !to_ptr(a[0], &c) || !to_size(a[1], &layer) || !to_ptr(a[2], &x) || !to_size(a[3], &m) || !to_ptr(a[7], &y)) return nullptr;
    if (!plan.get(a[4], "lLqQ", 8) || !tok.get(a[5], "i", 4) || !w.get(a[6], "f", 4) || plan.count() % 3 != 0 || w.count() < tok.count()) Py_RETURN_NONE;
    ALLOW(smx_moe_layer_dev(c, layer, x, m, (const size_t*)plan.b.buf, plan.count() / 3, (const int32_t*)tok.b.buf, (const float*)w.b.buf, tok.count(), y));
}
// (ctx, layer, xs, m, plan, slot_tok, wslot, y): host rows
FN(moe_layer) {
    smx_ctx* c; size_t layer, m; Array x, y, plan, tok, w;
    if (!argc_is(n, 8) || !to_ptr(a[0], &c) || !to_size(a[1], &layer) || !to_size(a[3], &m)) return nullptr;
    if (!x.get(a[2], "f", 4) || !plan.get(a[4], "lLqQ", 8) || !tok.get(a[5], "i", 4) || !w.get(a[6], "f", 4) || !y.get(a[7], "f", 4, true) ||
        plan.count() % 3 != 0 || w.count() < tok.count()) Py_RETURN_NONE;
    ALLOW(smx_moe_layer(c, layer, (const float*)x.b.buf, m, (const size_t*)plan.b.buf, plan.count() / 3, (const int32_t*)tok.b.buf,
                        (const float*)w.b.buf, tok.count(), (float*)y.b.buf, y.count()));
}

#define M(name, fn) {name, (PyCFunction)(void (*)(void))(fn), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    M("gemv_dev", rows_dev<smx_gemv_dev>), M("gemm_dev", rows_dev<smx_gemm_dev>), M("gemv_noalloc_dev", rows_dev<smx_gemv_noalloc_dev>),
    M("gemv_f32_dev", gemv_f32_dev), M("gemm_fused_dev", gemm_fused_dev), M("ffn_gate_up_dev", ffn_gate_up_dev),
    M("gemv_batch_dev", gemv_batch_dev), M("gemv_fused_dev", gemv_fused_dev), M("moe_route_dev", moe_route_dev),
    M("moe_ffn_logits_dev", moe_ffn_logits_dev), M("moe_ffn_routed_dev", moe_ffn_routed_dev), M("graph_launch", graph_launch),
    M("gemv", gemv_host<smx_gemv>), M("gemv_f32", gemv_host<smx_gemv_f32>), M("gemv_rows", rows_host<smx_gemv_rows>), M("gemm", rows_host<smx_gemm>),
    M("lm_head_argmax_rows", lm_head_argmax_rows), M("gemv_batch", gemv_batch), M("moe_ffn", moe_ffn), M("moe_ffn_dev", moe_ffn_dev),
    M("moe_layer_dev", moe_layer_dev), M("moe_layer", moe_layer), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_smx_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__smx_native(void) { return PyModule_Create(&module); }
