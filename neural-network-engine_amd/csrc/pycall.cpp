// CPython module nne_pycall: the calls of a decode or prefill step from Python
// to the C ABI (include/nne_attn.h) without ctypes.
//
// A small call's GPU time is 6-13 us; converting its 18-25 arguments through
// ctypes took 4-5 us of host time and building its shape arrays 3 us more, so a
// loop of such calls ran at the host's pace.  Here the arguments are read
// straight from Python ints and tuples.  Host time per call: a prefill of 256
// rows 15.4 -> 8.3 us (10.5 with ctypes on plain addresses), a decode step of one
// sequence 19.2 -> 9.7 (12.7).
//
// Each function takes the address of its ABI function first (the package loads
// the library and owns it) and returns the ABI's status.  Shapes and strides
// are tuples of 4 ints, device pointers ints or None, host arrays any object
// with a contiguous buffer or None, a workspace the tuple (records,
// records_bytes, counters, n_counters) or None.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "nne_attn.h"

namespace {

// Reads the arguments in order; after the first bad one the error is set and
// every later read returns zeros.
struct Args {
    PyObject* const* a;
    Py_ssize_t n, i = 0;
    bool ok = true;
    Py_buffer host[1];
    int n_host = 0;

    Args(PyObject* const* args, Py_ssize_t count) : a(args), n(count) {}
    ~Args() {
        for (int k = 0; k < n_host; ++k) PyBuffer_Release(&host[k]);
    }
    PyObject* next() {
        if (!ok) return nullptr;
        if (i < n) return a[i++];
        PyErr_SetString(PyExc_TypeError, "nne_pycall: too few arguments");
        ok = false;
        return nullptr;
    }
    int64_t integer() {
        PyObject* o = next();
        if (!o) return 0;
        const long long v = PyLong_AsLongLong(o);
        if (v == -1 && PyErr_Occurred()) ok = false;
        return v;
    }
    template <typename T>
    T* pointer() {
        PyObject* o = next();
        if (!o || o == Py_None) return nullptr;
        void* p = PyLong_AsVoidPtr(o);
        if (!p && PyErr_Occurred()) ok = false;
        return static_cast<T*>(p);
    }
    float real() {
        PyObject* o = next();
        if (!o) return 0.f;
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) ok = false;
        return (float)v;
    }
    void ints(PyObject* o, int64_t* out) {
        if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 4) {
            PyErr_SetString(PyExc_TypeError, "nne_pycall: expected a tuple of 4 ints");
            ok = false;
            return;
        }
        for (int k = 0; k < 4; ++k) {
            out[k] = PyLong_AsLongLong(PyTuple_GET_ITEM(o, k));
            if (out[k] == -1 && PyErr_Occurred()) { ok = false; return; }
        }
    }
    struct Dims { int64_t v[4] = {0, 0, 0, 0}; };
    Dims dims() {
        Dims d;
        if (PyObject* o = next()) ints(o, d.v);
        return d;
    }
    int32_t* host_array() {
        PyObject* o = next();
        if (!o || o == Py_None) return nullptr;
        if (PyObject_GetBuffer(o, &host[n_host], PyBUF_SIMPLE) != 0) {
            ok = false;
            return nullptr;
        }
        return static_cast<int32_t*>(host[n_host++].buf);
    }
    nne_workspace_t ws_store;
    const nne_workspace_t* workspace() {
        PyObject* o = next();
        if (!o || o == Py_None) return nullptr;
        int64_t v[4] = {0, 0, 0, 0};
        ints(o, v);
        ws_store.records = reinterpret_cast<void*>((uintptr_t)v[0]);
        ws_store.records_bytes = (uint64_t)v[1];
        ws_store.counters = reinterpret_cast<uint32_t*>((uintptr_t)v[2]);
        ws_store.n_counters = (uint64_t)v[3];
        return &ws_store;
    }
    bool done() {
        if (ok && i != n) {
            PyErr_SetString(PyExc_TypeError, "nne_pycall: too many arguments");
            ok = false;
        }
        return ok;
    }
};

template <typename F>
F* function(Args& a) {
    F* f = reinterpret_cast<F*>(a.pointer<void>());
    if (a.ok && !f) {
        PyErr_SetString(PyExc_ValueError, "nne_pycall: null function");
        a.ok = false;
    }
    return f;
}

PyObject* flash(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Args a(args, n);
    auto* f = function<decltype(nne_flash_attention_forward_ws)>(a);
    auto* q = a.pointer<const float>();
    const auto qs = a.dims(), qst = a.dims();
    auto* k = a.pointer<const float>();
    const auto ks = a.dims(), kst = a.dims();
    auto* v = a.pointer<const float>();
    const auto vs = a.dims(), vst = a.dims();
    auto* o = a.pointer<float>();
    const auto ost = a.dims();
    const int causal = (int)a.integer(), has_scale = (int)a.integer();
    const float scale = a.real();
    const int64_t br = a.integer(), bc = a.integer();
    const nne_workspace_t* ws = a.workspace();
    void* stream = a.pointer<void>();
    if (!a.done()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(q, qs.v, qst.v, k, ks.v, kst.v, v, vs.v, vst.v, o, ost.v, causal, has_scale, scale, br, bc,
           ws, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Args a(args, n);
    auto* f = function<decltype(nne_attention_forward_ws)>(a);
    auto* q = a.pointer<const float>();
    const auto qs = a.dims(), qst = a.dims();
    auto* k = a.pointer<const float>();
    const auto ks = a.dims(), kst = a.dims();
    auto* v = a.pointer<const float>();
    const auto vs = a.dims(), vst = a.dims();
    auto* o = a.pointer<float>();
    const auto ost = a.dims();
    const int causal = (int)a.integer();
    const int64_t q_offset = a.integer();
    const int has_scale = (int)a.integer();
    const float scale = a.real();
    const nne_workspace_t* ws = a.workspace();
    void* stream = a.pointer<void>();
    if (!a.done()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(q, qs.v, qst.v, k, ks.v, kst.v, v, vs.v, vst.v, o, ost.v, causal, q_offset, has_scale, scale,
           ws, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

PyObject* decode_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Args a(args, n);
    auto* f = function<decltype(nne_decode_attention)>(a);
    auto* q = a.pointer<const float>();
    const auto qst = a.dims();
    auto *kc = a.pointer<const float>(), *vc = a.pointer<const float>();
    auto* lens = a.pointer<const int32_t>();
    const int32_t* lens_host = a.host_array();
    auto* o = a.pointer<float>();
    const auto ost = a.dims();
    const int64_t B = a.integer(), Hq = a.integer(), Hkv = a.integer(), cap = a.integer(), d = a.integer();
    const int has_scale = (int)a.integer();
    const float scale = a.real();
    const nne_workspace_t* ws = a.workspace();
    void* stream = a.pointer<void>();
    if (!a.done()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(q, qst.v, kc, vc, lens, lens_host, o, ost.v, B, Hq, Hkv, cap, d, has_scale, scale, ws, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

PyObject* decode_step(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Args a(args, n);
    auto* f = function<decltype(nne_decode_step)>(a);
    auto* q = a.pointer<const float>();
    const auto qst = a.dims();
    auto *kc = a.pointer<float>(), *vc = a.pointer<float>();
    auto* lens = a.pointer<int32_t>();
    int32_t* lens_host = a.host_array();
    auto* kn = a.pointer<const float>();
    const auto knst = a.dims();
    auto* vn = a.pointer<const float>();
    const auto vnst = a.dims();
    auto* o = a.pointer<float>();
    const auto ost = a.dims();
    const int64_t B = a.integer(), Hq = a.integer(), Hkv = a.integer(), cap = a.integer(), d = a.integer();
    const int has_scale = (int)a.integer();
    const float scale = a.real();
    const nne_workspace_t* ws = a.workspace();
    void* stream = a.pointer<void>();
    if (!a.done()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(q, qst.v, kc, vc, lens, lens_host, kn, knst.v, vn, vnst.v, o, ost.v, B, Hq, Hkv, cap, d,
           has_scale, scale, ws, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

PyObject* qkv_rope(PyObject*, PyObject* const* args, Py_ssize_t n) {
    Args a(args, n);
    auto* f = function<decltype(nne_qkv_rope_ws)>(a);
    auto* x = a.pointer<const float>();
    const int64_t x_rs = a.integer();
    auto* w = a.pointer<const float>();
    auto *bq = a.pointer<const float>(), *bk = a.pointer<const float>(), *bv = a.pointer<const float>();
    auto *cos = a.pointer<const float>(), *sin = a.pointer<const float>();
    const int64_t max_seq = a.integer(), table_d = a.integer();
    auto* pos = a.pointer<const int32_t>();
    const int32_t* pos_host = a.host_array();
    auto *q = a.pointer<float>(), *k = a.pointer<float>(), *v = a.pointer<float>();
    const int64_t B = a.integer(), C = a.integer(), Hq = a.integer(), Hkv = a.integer(), d = a.integer();
    const nne_workspace_t* ws = a.workspace();
    void* stream = a.pointer<void>();
    if (!a.done()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(x, x_rs, w, bq, bk, bv, cos, sin, max_seq, table_d, pos, pos_host, q, k, v, B, C, Hq, Hkv, d,
           ws, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

#define NNE_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {NNE_METHOD(flash), NNE_METHOD(attention), NNE_METHOD(decode_attention),
                         NNE_METHOD(decode_step), NNE_METHOD(qkv_rope), {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "nne_pycall", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_nne_pycall(void) { return PyModule_Create(&module); }
