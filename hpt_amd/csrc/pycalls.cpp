// The calls of the tensor API that return a fresh tensor, from the interpreter straight into the C ABI: the views are read
// from the tensor's attributes, the result's shape, dtype and memory are found, and the operator is queued, in one
// crossing. Through ctypes each of these was a crossing of its own with its arrays built as Python objects: 13.1 us for a
// sum and 11.0 us for a softmax of which the library's own share is 3.6 and 4.3.
//
// Nothing is decided here: shapes, dtypes, memory and errors come from the same entry points as before. A call that this
// file does not take (more than 32 dims, values that are no 64-bit integers) returns None and the caller goes the long way.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "hpt_hip.h"

namespace {

constexpr int kRank = 32;
constexpr size_t kAlign = 64;  // of every tensor's memory

PyObject *s_ptr, *s_shape, *s_strides, *s_dtype, *s_code, *s_device;

struct View {
    hpt_view v;
    int64_t shape[kRank], strides[kRank];
};

// Integers of a list; the number of them, or -1 for anything else.
int integers(PyObject* list, int64_t* out) {
    if (!PyList_Check(list) || PyList_GET_SIZE(list) > kRank) return -1;
    const int n = (int)PyList_GET_SIZE(list);
    for (int i = 0; i < n; ++i) {
        PyObject* o = PyList_GET_ITEM(list, i);
        if (!PyLong_Check(o)) return -1;
        int overflow = 0;
        out[i] = PyLong_AsLongLongAndOverflow(o, &overflow);
        if (overflow) return -1;
    }
    return n;
}

// An attribute that is an integer; false for anything else (no exception is left behind).
bool integer(PyObject* o, PyObject* name, int64_t* out) {
    PyObject* a = PyObject_GetAttr(o, name);
    if (!a) {
        PyErr_Clear();
        return false;
    }
    bool ok = PyLong_Check(a);
    if (ok) {
        *out = (int64_t)PyLong_AsUnsignedLongLongMask(a);
        if (PyErr_Occurred()) {
            PyErr_Clear();
            ok = false;
        }
    }
    Py_DECREF(a);
    return ok;
}

bool dims(PyObject* o, PyObject* name, int64_t* out, int* n) {
    PyObject* a = PyObject_GetAttr(o, name);
    if (!a) {
        PyErr_Clear();
        return false;
    }
    *n = integers(a, out);
    Py_DECREF(a);
    return *n >= 0;
}

bool view_of(PyObject* t, View* w) {
    int64_t ptr, code;
    int n, m;
    if (!integer(t, s_ptr, &ptr) || !dims(t, s_shape, w->shape, &n) || !dims(t, s_strides, w->strides, &m) || n != m) return false;
    PyObject* d = PyObject_GetAttr(t, s_dtype);
    if (!d) {
        PyErr_Clear();
        return false;
    }
    const bool ok = integer(d, s_code, &code);
    Py_DECREF(d);
    if (!ok) return false;
    w->v.data = (void*)ptr;
    w->v.shape = w->shape;
    w->v.strides = w->strides;
    w->v.ndim = n;
    w->v.dtype = (int32_t)code;
    return true;
}

// A contiguous result of the given shape: memory for it, and its view.
struct Result {
    View w;
    size_t bytes = 0;
    void* p = nullptr;
    int32_t device = 0;
    bool ordered = false;

    int32_t allocate(int32_t dev, uint64_t stream, int32_t dtype, int ndim) {
        uint64_t s = 1;
        for (int i = ndim - 1; i >= 0; --i) {
            w.strides[i] = (int64_t)s;
            s *= (uint64_t)w.shape[i];
        }
        device = dev;
        bytes = (size_t)s * hpt_hip_dtype_size(dtype);
        // (a result whose first use is queued on the default stream may be memory that earlier work there still uses)
        ordered = stream == 0;
        const int32_t st = ordered ? hpt_hip_alloc_ordered(dev, bytes, kAlign, &p) : hpt_hip_alloc(dev, bytes, kAlign, 0, &p);
        w.v = hpt_view{p, w.shape, w.strides, ndim, dtype};
        return st;
    }
    // The operator was refused. (Memory that earlier work on the default stream still uses stays that until somebody waits.)
    void release() {
        if (p && ordered) (void)hpt_hip_free_ordered(device, p, bytes, kAlign);
        else if (p) (void)hpt_hip_free(device, p, bytes, kAlign);
        p = nullptr;
    }
};

PyObject* list_of(const int64_t* v, int n) {
    PyObject* l = PyList_New(n);
    for (int i = 0; l && i < n; ++i) {
        PyObject* o = PyLong_FromLongLong(v[i]);
        if (!o) {
            Py_CLEAR(l);
            break;
        }
        PyList_SET_ITEM(l, i, o);
    }
    return l;
}

// (address, bytes, shape, strides, dtype code) of a result that has been queued, its shape as the caller wants it
PyObject* answer(Result& r, const int64_t* shape, int ndim) {
    int64_t strides[kRank];
    uint64_t s = 1;
    for (int i = ndim - 1; i >= 0; --i) {
        strides[i] = (int64_t)s;
        s *= (uint64_t)shape[i];
    }
    PyObject* a = list_of(shape, ndim);
    PyObject* b = a ? list_of(strides, ndim) : nullptr;
    PyObject* t = b ? Py_BuildValue("KnNNi", (unsigned long long)(uintptr_t)r.p, (Py_ssize_t)r.bytes, a, b, (int)r.w.v.dtype) : nullptr;
    if (!t) {
        if (!b) Py_XDECREF(a);
        // (out of memory on the host: the queued operator still writes the block, so it is given back behind it)
        (void)hpt_hip_device_synchronize(r.device);
        r.release();
    }
    return t;
}

PyObject* status(int32_t s) { return PyLong_FromLong(s); }

bool wrong_count(Py_ssize_t n, Py_ssize_t want) {
    if (n == want) return false;
    PyErr_Format(PyExc_TypeError, "%zd arguments wanted, got %zd", want, n);
    return true;
}

// The arguments every call starts with: tensor, stream.
bool opening(PyObject* const* a, View* in, int32_t* dev, uint64_t* stream) {
    int64_t d;
    if (!PyLong_Check(a[1]) || !view_of(a[0], in) || !integer(a[0], s_device, &d)) return false;
    *stream = PyLong_AsUnsignedLongLongMask(a[1]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    *dev = (int32_t)d;
    return true;
}

// reduce(tensor, stream, op, axes, keep_dims)
PyObject* py_reduce(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (wrong_count(n, 5)) return nullptr;
    View in;
    int32_t dev;
    uint64_t stream;
    int64_t axes[kRank];
    if (!opening(a, &in, &dev, &stream)) Py_RETURN_NONE;
    const long op = PyLong_AsLong(a[2]);
    const int naxes = integers(a[3], axes), keep = PyObject_IsTrue(a[4]);
    if (PyErr_Occurred()) return nullptr;
    if (naxes < 0) Py_RETURN_NONE;
    Result r;
    int64_t shape[kRank];
    int32_t od = 0, nd = 0, sd = 0, st;
    Py_BEGIN_ALLOW_THREADS
    st = hpt_hip_reduce_out_dtype((int32_t)op, in.v.dtype, &od);
    if (st == HPT_OK) st = hpt_hip_reduce_shape(in.shape, in.v.ndim, axes, naxes, 0, r.w.shape, &nd);
    if (st == HPT_OK && keep) st = hpt_hip_reduce_shape(in.shape, in.v.ndim, axes, naxes, 1, shape, &sd);
    if (st == HPT_OK) st = r.allocate(dev, stream, od, nd);
    if (st == HPT_OK) {
        st = hpt_hip_reduce(dev, (void*)stream, (int32_t)op, &in.v, axes, naxes, 1, &r.w.v);
        if (st != HPT_OK) r.release();
    }
    Py_END_ALLOW_THREADS
    if (st != HPT_OK) return status(st);
    return keep ? answer(r, shape, sd) : answer(r, r.w.shape, nd);
}

// argreduce(tensor, stream, is_max, axes of one, keep_dims)
PyObject* py_argreduce(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (wrong_count(n, 5)) return nullptr;
    View in;
    int32_t dev;
    uint64_t stream;
    int64_t axes[kRank];
    if (!opening(a, &in, &dev, &stream)) Py_RETURN_NONE;
    const int is_max = PyObject_IsTrue(a[2]), naxes = integers(a[3], axes), keep = PyObject_IsTrue(a[4]);
    if (PyErr_Occurred()) return nullptr;
    if (naxes != 1) Py_RETURN_NONE;
    Result r;
    int64_t shape[kRank];
    int32_t nd = 0, sd = 0, st;
    Py_BEGIN_ALLOW_THREADS
    st = hpt_hip_reduce_shape(in.shape, in.v.ndim, axes, 1, 0, r.w.shape, &nd);
    if (st == HPT_OK && keep) st = hpt_hip_reduce_shape(in.shape, in.v.ndim, axes, 1, 1, shape, &sd);
    if (st == HPT_OK) st = r.allocate(dev, stream, HPT_I64, nd);
    if (st == HPT_OK) {
        st = hpt_hip_argreduce(dev, (void*)stream, is_max, &in.v, axes[0], &r.w.v);
        if (st != HPT_OK) r.release();
    }
    Py_END_ALLOW_THREADS
    if (st != HPT_OK) return status(st);
    return keep ? answer(r, shape, sd) : answer(r, r.w.shape, nd);
}

// A result of the input's shape, in the dtype of the float-valued operators.
int32_t allocate_like(Result& r, const View& in, int32_t dev, uint64_t stream) {
    int32_t od = 0;
    const int32_t st = hpt_hip_reduce_out_dtype(HPT_MEAN, in.v.dtype, &od);
    if (st != HPT_OK) return st;
    for (int i = 0; i < in.v.ndim; ++i) r.w.shape[i] = in.shape[i];
    return r.allocate(dev, stream, od, in.v.ndim);
}

// softmax(tensor, stream, log, axis)
PyObject* py_softmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (wrong_count(n, 4)) return nullptr;
    View in;
    int32_t dev;
    uint64_t stream;
    if (!opening(a, &in, &dev, &stream)) Py_RETURN_NONE;
    const int log = PyObject_IsTrue(a[2]);
    int overflow = 0;
    const long long axis = PyLong_AsLongLongAndOverflow(a[3], &overflow);
    if (PyErr_Occurred()) return nullptr;
    if (overflow) Py_RETURN_NONE;
    Result r;
    int32_t st;
    Py_BEGIN_ALLOW_THREADS
    st = allocate_like(r, in, dev, stream);
    if (st == HPT_OK) {
        st = hpt_hip_softmax(dev, (void*)stream, log, &in.v, axis, &r.w.v);
        if (st != HPT_OK) r.release();
    }
    Py_END_ALLOW_THREADS
    return st != HPT_OK ? status(st) : answer(r, r.w.shape, in.v.ndim);
}

// layernorm(tensor, stream, normalized dims, gamma, beta, eps, residual): the last four may be None
PyObject* py_layernorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (wrong_count(n, 7)) return nullptr;
    View in, g, b, res;
    int32_t dev;
    uint64_t stream;
    if (!opening(a, &in, &dev, &stream)) Py_RETURN_NONE;
    const long nn = PyLong_AsLong(a[2]);
    const double eps = PyFloat_AsDouble(a[5]);
    if (PyErr_Occurred()) return nullptr;
    const bool have_g = a[3] != Py_None, have_b = a[4] != Py_None, have_r = a[6] != Py_None;
    if ((have_g && !view_of(a[3], &g)) || (have_b && !view_of(a[4], &b)) || (have_r && !view_of(a[6], &res))) Py_RETURN_NONE;
    const hpt_view *gv = have_g ? &g.v : nullptr, *bv = have_b ? &b.v : nullptr;
    Result r;
    int32_t st;
    Py_BEGIN_ALLOW_THREADS
    st = allocate_like(r, in, dev, stream);
    if (st == HPT_OK) {
        st = have_r ? hpt_hip_add_layernorm(dev, (void*)stream, &in.v, &res.v, (int32_t)nn, gv, bv, eps, &r.w.v)
                    : hpt_hip_layernorm(dev, (void*)stream, &in.v, (int32_t)nn, gv, bv, eps, &r.w.v);
        if (st != HPT_OK) r.release();
    }
    Py_END_ALLOW_THREADS
    return st != HPT_OK ? status(st) : answer(r, r.w.shape, in.v.ndim);
}

// softmax_causal(tensor, stream, log, scale, offset)
PyObject* py_softmax_causal(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (wrong_count(n, 5)) return nullptr;
    View in;
    int32_t dev;
    uint64_t stream;
    if (!opening(a, &in, &dev, &stream)) Py_RETURN_NONE;
    const int log = PyObject_IsTrue(a[2]);
    const double scale = PyFloat_AsDouble(a[3]);
    int overflow = 0;
    const long long offset = PyLong_AsLongLongAndOverflow(a[4], &overflow);
    if (PyErr_Occurred()) return nullptr;
    if (overflow) Py_RETURN_NONE;
    Result r;
    int32_t st;
    Py_BEGIN_ALLOW_THREADS
    for (int i = 0; i < in.v.ndim; ++i) r.w.shape[i] = in.shape[i];
    st = r.allocate(dev, stream, in.v.dtype, in.v.ndim);
    if (st == HPT_OK) {
        st = hpt_hip_softmax_causal(dev, (void*)stream, log, &in.v, scale, offset, &r.w.v);
        if (st != HPT_OK) r.release();
    }
    Py_END_ALLOW_THREADS
    return st != HPT_OK ? status(st) : answer(r, r.w.shape, in.v.ndim);
}

// free(device, address, bytes, ordered) -> status
PyObject* py_free(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (wrong_count(n, 4)) return nullptr;
    const long dev = PyLong_AsLong(a[0]);
    const unsigned long long p = PyLong_AsUnsignedLongLong(a[1]);
    const unsigned long long bytes = PyLong_AsUnsignedLongLong(a[2]);
    const int ordered = PyObject_IsTrue(a[3]);
    if (PyErr_Occurred()) return nullptr;
    int32_t st;
    Py_BEGIN_ALLOW_THREADS
    st = ordered ? hpt_hip_free_ordered((int32_t)dev, (void*)(uintptr_t)p, (size_t)bytes, kAlign)
                 : hpt_hip_free((int32_t)dev, (void*)(uintptr_t)p, (size_t)bytes, kAlign);
    Py_END_ALLOW_THREADS
    return status(st);
}

#define HPT_CALL(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {HPT_CALL("reduce", py_reduce),
                         HPT_CALL("argreduce", py_argreduce),
                         HPT_CALL("softmax", py_softmax),
                         HPT_CALL("layernorm", py_layernorm),
                         HPT_CALL("softmax_causal", py_softmax_causal),
                         HPT_CALL("free", py_free),
                         {nullptr, nullptr, 0, nullptr}};
#undef HPT_CALL

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
    s_ptr = PyUnicode_InternFromString("ptr");
    s_shape = PyUnicode_InternFromString("shape");
    s_strides = PyUnicode_InternFromString("strides");
    s_dtype = PyUnicode_InternFromString("dtype");
    s_code = PyUnicode_InternFromString("code");
    s_device = PyUnicode_InternFromString("device");
    if (!s_ptr || !s_shape || !s_strides || !s_dtype || !s_code || !s_device) return nullptr;
    return PyModule_Create(&module);
}
