// pyhost.cpp -- the host side of one call from Python: Matrix operands to descriptors, the C entry point, its status.
//
// A small call is bound by its host side.  Through ctypes a two-operand call takes 5.3 us, 2.3 of them the launch: the
// descriptors are packed by Python code (0.4 us each) and converted argument by argument.  Here the attributes of the
// Matrix objects are read once, straight into zenu_tensor_t (3.3 us in all); the optimizers' argument arrays, four
// pointers and a size per tensor, are filled the same way (0.3 us per tensor, 1.5 before).
//
// Every function takes exactly the forms that programs pass all the time -- Matrix itself (no subclass), float32 or
// float64, tuples of plain integers, plain numbers, a stream as None, an integer or a c_void_p -- and returns True when it
// has made the call, False when it has not looked further than an operand of another form: the caller then goes the
// ctypes way, which accepts, converts and refuses as it always did.  A status that is not OK is raised by _lib.check.
// Nothing is kept between calls but the addresses of the entry points.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>

#include <climits>
#include <new>
#include <vector>

#include "../../include/zenu_hip.h"

namespace {

PyTypeObject *g_matrix = nullptr, *g_void_p = nullptr;
PyObject *g_f32 = nullptr, *g_f64 = nullptr, *g_check = nullptr;
PyObject *s_buf, *s_offset, *s_shape, *s_stride, *s_dtype, *s_ptr, *s_value;

#define ZENU_PY_ENTRIES(X)                                                                                     \
    X(binary) X(binary_assign) X(binary_scalar) X(binary_scalar_assign) X(unary) X(copy) X(broadcast) X(relu)  \
    X(relu_backward) X(tanh_backward) X(sigmoid_backward) X(relu_backward_bias_grad) X(softmax)                \
    X(bias_add_relu) X(sum_to) X(adam_step_multi) X(sgd_step_multi)
struct Entries {
#define X(name) decltype(&zenu_hip_##name) name;
    ZENU_PY_ENTRIES(X)
#undef X
} g = {};
bool g_bound = false;

// ---- arguments ---------------------------------------------------------------------------------------------
// Each returns false, without an exception set, for a form that is left to the general path.

bool as_int64(PyObject *o, int64_t &v)
{
    if (!o || !PyLong_CheckExact(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return !overflow;
}

bool as_int(PyObject *o, int &v)
{
    int64_t w;
    if (!as_int64(o, w) || w < INT_MIN || w > INT_MAX) return false;
    v = (int)w;
    return true;
}

bool as_double(PyObject *o, double &v)
{
    if (PyFloat_CheckExact(o)) {
        v = PyFloat_AS_DOUBLE(o);
        return true;
    }
    int64_t w;
    if (!as_int64(o, w) || w > (1ll << 53) || w < -(1ll << 53)) return false;
    v = (double)w;
    return true;
}

bool as_address(PyObject *o, uintptr_t &v)
{
    if (!o || !PyLong_CheckExact(o)) return false;
    v = (uintptr_t)PyLong_AsUnsignedLongLong(o);
    if (v == (uintptr_t)-1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

bool as_stream(PyObject *o, zenu_stream_t &s)
{
    uintptr_t v = 0;
    if (o == Py_None) {
        s = nullptr;
        return true;
    }
    if (Py_TYPE(o) == g_void_p) {
        PyObject *value = PyObject_GetAttr(o, s_value);
        if (!value) {
            PyErr_Clear();
            return false;
        }
        const bool ok = value == Py_None || as_address(value, v);
        Py_DECREF(value);
        s = (zenu_stream_t)v;
        return ok;
    }
    if (!as_address(o, v)) return false;
    s = (zenu_stream_t)v;
    return true;
}

// The descriptor of a Matrix and its dtype code (a zenu_dtype); elements of dtypes without a code are left to the general path.
bool as_tensor(PyObject *m, zenu_tensor_t &t, int &code)
{
    if (Py_TYPE(m) != g_matrix) return false;
    PyObject **dict = _PyObject_GetDictPtr(m);
    if (!dict || !*dict) return false;
    auto get = [&](PyObject *name) {
        PyObject *v = PyDict_GetItemWithError(*dict, name);   // borrowed
        if (!v) PyErr_Clear();
        return v;
    };
    PyObject *dtype = get(s_dtype), *shape = get(s_shape), *stride = get(s_stride), *buf = get(s_buf);
    int64_t offset;
    if (dtype == g_f32) code = ZENU_F32;
    else if (dtype == g_f64) code = ZENU_F64;
    else return false;
    if (!shape || !stride || !buf || !PyTuple_CheckExact(shape) || !PyTuple_CheckExact(stride)) return false;
    const Py_ssize_t n = PyTuple_GET_SIZE(shape);
    if (n > ZENU_MAX_DIM || PyTuple_GET_SIZE(stride) != n || !as_int64(get(s_offset), offset) || offset < 0) return false;
    t.ndim = (int32_t)n;
    t.reserved = 0;
    for (Py_ssize_t i = 0; i < ZENU_MAX_DIM; i++) t.shape[i] = t.stride[i] = 0;
    for (Py_ssize_t i = 0; i < n; i++) {
        int64_t a, b;
        if (!as_int64(PyTuple_GET_ITEM(shape, i), a) || !as_int64(PyTuple_GET_ITEM(stride, i), b)) return false;
        t.shape[i] = a;
        t.stride[i] = b;
    }
    Py_INCREF(buf);   // (ptr may be a property: its code could take the buffer out of the Matrix)
    PyObject *ptr = PyObject_GetAttr(buf, s_ptr);
    Py_DECREF(buf);
    if (!ptr) {
        PyErr_Clear();
        return false;
    }
    uintptr_t address;
    const bool ok = as_address(ptr, address);
    Py_DECREF(ptr);
    if (!ok) return false;
    t.ptr = (void *)(address + (uintptr_t)offset * (code == ZENU_F32 ? 4 : 8));
    return true;
}

bool default_stride(const zenu_tensor_t &t)
{
    int64_t s = 1;
    for (int i = t.ndim - 1; i >= 0; i--) {
        if (t.stride[i] != s) return false;
        s *= t.shape[i];
    }
    return true;
}

// ---- a call ------------------------------------------------------------------------------------------------------

PyObject *finish(int status, const char *where)
{
    if (status == ZENU_OK) Py_RETURN_TRUE;
    PyObject *r = PyObject_CallFunction(g_check, "is", status, where);   // raises
    if (!r) return nullptr;
    Py_DECREF(r);
    Py_RETURN_TRUE;
}

// Operands in order, the first one's dtype code for the call (as in the general path), then the stream.
struct Operands {
    zenu_tensor_t t[4];
    int code = 0;
    zenu_stream_t stream = nullptr;
    bool ok = true;
    Operands(PyObject *const *args, int n, PyObject *s)
    {
        for (int i = 0; i < n && ok; i++) {
            int c;
            ok = as_tensor(args[i], t[i], c);
            if (i == 0) code = c;
        }
        ok = ok && as_stream(s, stream);
    }
};

template <typename Call> PyObject *run(const char *where, Call call)
{
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = call();
    Py_END_ALLOW_THREADS
    return finish(status, where);
}

#define ZENU_PY(name, nargs)                                                                     \
    PyObject *py_##name(PyObject *, PyObject *const *a, Py_ssize_t n)                            \
    {                                                                                            \
        if (n != (nargs)) {                                                                      \
            PyErr_SetString(PyExc_TypeError, #name ": wrong number of arguments");               \
            return nullptr;                                                                      \
        }                                                                                        \
        if (!g_bound) Py_RETURN_FALSE;
#define ZENU_PY_END }

ZENU_PY(binary, 5)   // op, to, lhs, rhs, stream
    int op;
    Operands o(a + 1, 3, a[4]);
    if (!o.ok || !as_int(a[0], op)) Py_RETURN_FALSE;
    return run("binary", [&] { return g.binary(op, o.code, &o.t[0], &o.t[1], &o.t[2], o.stream); });
ZENU_PY_END

ZENU_PY(binary_assign, 4)   // op, to, rhs, stream
    int op;
    Operands o(a + 1, 2, a[3]);
    if (!o.ok || !as_int(a[0], op)) Py_RETURN_FALSE;
    return run("binary_assign", [&] { return g.binary_assign(op, o.code, &o.t[0], &o.t[1], o.stream); });
ZENU_PY_END

ZENU_PY(binary_scalar, 5)   // op, to, other, scalar, stream
    int op;
    double s;
    Operands o(a + 1, 2, a[4]);
    if (!o.ok || !as_int(a[0], op) || !as_double(a[3], s)) Py_RETURN_FALSE;
    return run("binary_scalar", [&] { return g.binary_scalar(op, o.code, &o.t[0], &o.t[1], s, o.stream); });
ZENU_PY_END

ZENU_PY(binary_scalar_assign, 4)   // op, to, scalar, stream
    int op;
    double s;
    Operands o(a + 1, 1, a[3]);
    if (!o.ok || !as_int(a[0], op) || !as_double(a[2], s)) Py_RETURN_FALSE;
    return run("binary_scalar_assign", [&] { return g.binary_scalar_assign(op, o.code, &o.t[0], s, o.stream); });
ZENU_PY_END

ZENU_PY(unary, 4)   // fn, to, other, stream
    int fn;
    Operands o(a + 1, 2, a[3]);
    if (!o.ok || !as_int(a[0], fn)) Py_RETURN_FALSE;
    return run("unary", [&] { return g.unary(fn, o.code, &o.t[0], &o.t[1], o.stream); });
ZENU_PY_END

ZENU_PY(copy, 3)   // to, src, stream
    Operands o(a, 2, a[2]);
    if (!o.ok) Py_RETURN_FALSE;
    return run("copy_from", [&] { return g.copy(o.code, &o.t[0], &o.t[1], o.stream); });
ZENU_PY_END

ZENU_PY(broadcast, 3)   // to, source, stream
    Operands o(a, 2, a[2]);
    if (!o.ok) Py_RETURN_FALSE;
    return run("broadcast", [&] { return g.broadcast(o.code, &o.t[0], &o.t[1], o.stream); });
ZENU_PY_END

ZENU_PY(relu, 4)   // to, other, alpha, stream
    double alpha;
    Operands o(a, 2, a[3]);
    if (!o.ok || !as_double(a[2], alpha)) Py_RETURN_FALSE;
    return run("relu", [&] { return g.relu(o.code, &o.t[0], &o.t[1], alpha, o.stream); });
ZENU_PY_END

ZENU_PY(relu_backward, 5)   // gx, gy, x, alpha, stream
    double alpha;
    Operands o(a, 3, a[4]);
    if (!o.ok || !as_double(a[3], alpha)) Py_RETURN_FALSE;
    return run("relu_backward", [&] { return g.relu_backward(o.code, &o.t[0], &o.t[1], &o.t[2], alpha, o.stream); });
ZENU_PY_END

ZENU_PY(tanh_backward, 4)   // gx, gy, x, stream
    Operands o(a, 3, a[3]);
    if (!o.ok) Py_RETURN_FALSE;
    return run("tanh_backward", [&] { return g.tanh_backward(o.code, &o.t[0], &o.t[1], &o.t[2], o.stream); });
ZENU_PY_END

ZENU_PY(sigmoid_backward, 4)   // gx, gy, x, stream
    Operands o(a, 3, a[3]);
    if (!o.ok) Py_RETURN_FALSE;
    return run("sigmoid_backward", [&] { return g.sigmoid_backward(o.code, &o.t[0], &o.t[1], &o.t[2], o.stream); });
ZENU_PY_END

ZENU_PY(relu_backward_bias_grad, 6)   // gx, gbias, gy, x, alpha, stream
    double alpha;
    Operands o(a, 4, a[5]);
    if (!o.ok || !as_double(a[4], alpha)) Py_RETURN_FALSE;
    return run("relu_backward_bias_grad", [&] {
        return g.relu_backward_bias_grad(o.code, &o.t[0], &o.t[1], &o.t[2], &o.t[3], alpha, o.stream);
    });
ZENU_PY_END

ZENU_PY(softmax, 4)   // to, source, axis, stream
    int axis;
    Operands o(a, 2, a[3]);
    if (!o.ok || !as_int(a[2], axis)) Py_RETURN_FALSE;
    return run("softmax_assign", [&] { return g.softmax(o.code, &o.t[0], &o.t[1], axis, o.stream); });
ZENU_PY_END

ZENU_PY(bias_add_relu, 6)   // act, z, bias, alpha, pre or None, stream
    double alpha;
    zenu_tensor_t pre;
    int code;
    const bool with_pre = a[4] != Py_None;
    Operands o(a, 3, a[5]);
    if (!o.ok || !as_double(a[3], alpha) || (with_pre && !as_tensor(a[4], pre, code))) Py_RETURN_FALSE;
    return run("bias_add_relu", [&] {
        return g.bias_add_relu(o.code, with_pre ? &pre : nullptr, &o.t[0], &o.t[1], &o.t[2], alpha, o.stream);
    });
ZENU_PY_END

ZENU_PY(sum_to, 3)   // source, target, stream
    Operands o(a, 2, a[2]);
    if (!o.ok) Py_RETURN_FALSE;
    return run("sum_to", [&] { return g.sum_to(o.code, &o.t[1], &o.t[0], o.stream); });
ZENU_PY_END

// ---- optimizers ----------------------------------------------------------------------------------------------------

// The tensors of an update in the order of the mapping: per entry with a gradient `kinds` matrices of one dtype in default
// stride.  Reading a matrix can run Python code (ptr may be a property, and another thread may get the GIL in it) that
// takes entries out of the mapping or of a dictionary of moments, so everything is held first and read afterwards; the
// matrices stay held while the GIL is released, as the argument lists of the general path hold them.
struct Update {
    std::vector<void *> ptr[4];
    std::vector<int64_t> sizes;
    std::vector<int32_t> decay;
    std::vector<PyObject *> held;
    int code = -1;
    ~Update() { for (PyObject *o : held) Py_DECREF(o); }

    void hold(PyObject *o)
    {
        held.push_back(o);
        Py_INCREF(o);
    }
    bool add(PyObject *const *matrices, int kinds)
    {
        zenu_tensor_t t;
        for (int k = 0; k < kinds; k++) {
            int c;
            if (!as_tensor(matrices[k], t, c) || !default_stride(t)) return false;
            if (code < 0) code = c;
            if (c != code) return false;
            ptr[k].push_back(t.ptr);
            if (k == 0) {
                int64_t n = 1;
                for (int i = 0; i < t.ndim; i++) n *= t.shape[i];
                sizes.push_back(n);
            }
        }
        return true;
    }
    // parameters: name -> (parameter, gradient or None).  m, v: name -> moment, or null.  weights: a set, or None.
    bool collect(PyObject *parameters, PyObject *m, PyObject *v, PyObject *weights)
    {
        if (!PyDict_CheckExact(parameters) || (m && (!PyDict_CheckExact(m) || !PyDict_CheckExact(v)))) return false;
        if (weights && weights != Py_None && !PyAnySet_CheckExact(weights)) return false;
        const size_t most = (size_t)PyDict_GET_SIZE(parameters);
        for (auto &p : ptr) p.reserve(most);
        sizes.reserve(most);
        decay.reserve(most);
        held.reserve((m ? 5 : 3) * most);
        PyObject *key, *value;
        Py_ssize_t at = 0;
        while (PyDict_Next(parameters, &at, &key, &value)) {   // nothing in this loop runs Python code
            if (!PyUnicode_CheckExact(key) || !PyTuple_CheckExact(value) || PyTuple_GET_SIZE(value) != 2) return false;
            if (PyTuple_GET_ITEM(value, 1) == Py_None) continue;
            hold(key);
            hold(PyTuple_GET_ITEM(value, 0));
            hold(PyTuple_GET_ITEM(value, 1));
        }
        const size_t entries = held.size() / 3;
        if (m) {
            for (size_t e = 0; e < entries; e++) {
                for (PyObject *moments : {m, v}) {
                    PyObject *moment = PyDict_GetItemWithError(moments, held[3 * e]);
                    if (!moment) {
                        PyErr_Clear();
                        return false;
                    }
                    hold(moment);
                }
            }
        }
        for (size_t e = 0; e < entries; e++) {
            PyObject *matrices[4] = {held[3 * e + 1], held[3 * e + 2], nullptr, nullptr};
            if (m) {
                matrices[2] = held[3 * entries + 2 * e];
                matrices[3] = held[3 * entries + 2 * e + 1];
            }
            if (!add(matrices, m ? 4 : 2)) return false;
            int in = 0;
            if (weights && weights != Py_None) in = PySet_Contains(weights, held[3 * e]);
            if (in < 0) {
                PyErr_Clear();
                return false;
            }
            decay.push_back(in);
        }
        return entries <= (size_t)INT_MAX;
    }
};

ZENU_PY(adam_step_multi, 11)   // parameters, m, v, weights or None, lr, beta1, beta2, epsilon, weight decay, step, stream
    double s[6];
    zenu_stream_t stream;
    for (int i = 0; i < 6; i++)
        if (!as_double(a[4 + i], s[i])) Py_RETURN_FALSE;
    if (!as_stream(a[10], stream)) Py_RETURN_FALSE;
    Update u;
    try {
        if (!u.collect(a[0], a[1], a[2], a[3])) Py_RETURN_FALSE;
    } catch (const std::bad_alloc &) {
        return PyErr_NoMemory();
    }
    if (u.sizes.empty()) Py_RETURN_TRUE;
    return run("adam_step_multi", [&] {
        return g.adam_step_multi(u.code, (int)u.sizes.size(), u.ptr[0].data(), u.ptr[1].data(), u.ptr[2].data(), u.ptr[3].data(),
                                 u.sizes.data(), s[0], s[1], s[2], s[3], s[4], u.decay.data(), s[5], stream);
    });
ZENU_PY_END

ZENU_PY(sgd_step_multi, 3)   // parameters, lr, stream
    double lr;
    zenu_stream_t stream;
    if (!as_double(a[1], lr) || !as_stream(a[2], stream)) Py_RETURN_FALSE;
    Update u;
    try {
        if (!u.collect(a[0], nullptr, nullptr, nullptr)) Py_RETURN_FALSE;
    } catch (const std::bad_alloc &) {
        return PyErr_NoMemory();
    }
    if (u.sizes.empty()) Py_RETURN_TRUE;
    return run("sgd_step_multi", [&] {
        return g.sgd_step_multi(u.code, (int)u.sizes.size(), u.ptr[0].data(), u.ptr[1].data(), u.sizes.data(), lr, stream);
    });
ZENU_PY_END

// ---- without a call --------------------------------------------------------------------------------------------------

// the bytes of a Matrix's zenu_tensor_t, or None for a form that is left to the general path
PyObject *py_pack(PyObject *, PyObject *m)
{
    zenu_tensor_t t;
    int code;
    if (!as_tensor(m, t, code)) Py_RETURN_NONE;
    return PyBytes_FromStringAndSize(reinterpret_cast<const char *>(&t), sizeof(t));
}

// the view of a Matrix with its last two axes exchanged, or None
PyObject *py_transpose(PyObject *, PyObject *m)
{
    if (Py_TYPE(m) != g_matrix) Py_RETURN_NONE;
    PyObject **dict = _PyObject_GetDictPtr(m);
    if (!dict || !*dict) Py_RETURN_NONE;
    PyObject *v[5], *names[5] = {s_buf, s_offset, s_shape, s_stride, s_dtype};
    for (int i = 0; i < 5; i++) {
        v[i] = PyDict_GetItemWithError(*dict, names[i]);
        if (!v[i]) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
    }
    for (int i = 2; i < 4; i++)
        if (!PyTuple_CheckExact(v[i]) || PyTuple_GET_SIZE(v[i]) < 2 || PyTuple_GET_SIZE(v[i]) != PyTuple_GET_SIZE(v[2])) Py_RETURN_NONE;
    for (PyObject *x : v) Py_INCREF(x);   // (an allocation can start the collector, whose finalizers may take them out of the Matrix)
    PyObject *view = g_matrix->tp_alloc(g_matrix, 0);
    bool ok = view != nullptr;
    for (int i = 2; i < 4 && ok; i++) {
        const Py_ssize_t n = PyTuple_GET_SIZE(v[i]);
        PyObject *turned = PyTuple_New(n);
        if (!turned) {
            ok = false;
            break;
        }
        for (Py_ssize_t k = 0; k < n; k++) {
            PyObject *e = PyTuple_GET_ITEM(v[i], k == n - 1 ? n - 2 : k == n - 2 ? n - 1 : k);
            Py_INCREF(e);
            PyTuple_SET_ITEM(turned, k, e);
        }
        Py_SETREF(v[i], turned);
    }
    for (int i = 0; i < 5 && ok; i++) ok = PyObject_SetAttr(view, names[i], v[i]) == 0;
    for (PyObject *x : v) Py_DECREF(x);
    if (!ok) {
        Py_XDECREF(view);
        return nullptr;
    }
    return view;
}

// setup(Matrix, c_void_p, dtype float32, dtype float64, check)
PyObject *py_setup(PyObject *, PyObject *args)
{
    PyObject *matrix, *void_p, *f32, *f64, *check;
    if (!PyArg_ParseTuple(args, "O!O!OOO", &PyType_Type, &matrix, &PyType_Type, &void_p, &f32, &f64, &check)) return nullptr;
    for (PyObject *o : {matrix, void_p, f32, f64, check}) Py_INCREF(o);
    g_matrix = reinterpret_cast<PyTypeObject *>(matrix);
    g_void_p = reinterpret_cast<PyTypeObject *>(void_p);
    g_f32 = f32;
    g_f64 = f64;
    g_check = check;
    Py_RETURN_NONE;
}

// bind(handle): the entry points of the loaded library, as dlopen returned it
PyObject *py_bind(PyObject *, PyObject *handle)
{
    void *h = PyLong_AsVoidPtr(handle);
    if (!h && PyErr_Occurred()) return nullptr;
    Entries e = {};
#define X(name)                                                                         \
    e.name = reinterpret_cast<decltype(e.name)>(dlsym(h, "zenu_hip_" #name));           \
    if (!e.name) {                                                                      \
        PyErr_SetString(PyExc_ImportError, "libzenu_hip.so has no zenu_hip_" #name);    \
        return nullptr;                                                                 \
    }
    ZENU_PY_ENTRIES(X)
#undef X
    g = e;
    g_bound = true;
    Py_RETURN_NONE;
}

#define M(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {
    ZENU_PY_ENTRIES(M)
    {"pack", py_pack, METH_O, nullptr},
    {"transpose", py_transpose, METH_O, nullptr},
    {"setup", py_setup, METH_VARARGS, nullptr},
    {"bind", py_bind, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
#undef M

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pyhost", "host side of zenu_amd's calls", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pyhost()
{
    struct { PyObject **p; const char *s; } names[] = {{&s_buf, "buf"}, {&s_offset, "offset"}, {&s_shape, "shape"}, {&s_stride, "stride"},
                                                        {&s_dtype, "dtype"}, {&s_ptr, "ptr"}, {&s_value, "value"}};
    for (auto &n : names)
        if (!(*n.p = PyUnicode_InternFromString(n.s))) return nullptr;
    return PyModule_Create(&module);
}
