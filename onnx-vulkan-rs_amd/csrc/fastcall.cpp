// CPython entry points for the calls that only enqueue: what ctypes does for them in about a microsecond (building a call
// from an argument list at run time) costs a tenth of that here, and a decode step or a small layer is bound by exactly
// this path -- one kernel launch is 2.2 us of host time, and the call around it was another 1.2 to 2.5.
//
// A function is bound by name to its address in the library the loader opened (this module is not linked against it);
// types come from include/hipcompute.h, so a change of a signature there is a compile error or a changed binding, never a
// mismatch. An argument of a pointer type may be None, a whole number (an address), a ctypes.c_void_p, a ctypes structure or
// a NumPy array; an argument this module cannot convert sends the call, as it came, to the ctypes function. As with ctypes, other Python threads run while the library works.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstddef>
#include <cstring>
#include <new>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/hipcompute.h"

namespace {

PyTypeObject *g_c_void_p, *g_structure, *g_ndarray;   // ctypes.c_void_p, ctypes.Structure, numpy.ndarray

// Conversions: false (no Python error set) when the value is not of a kind handled here. `view` holds a buffer for the call.
struct Views {
    Py_buffer held[8];
    int n = 0;
    ~Views() {
        while (n > 0) PyBuffer_Release(&held[--n]);
    }
};

bool to_integer(PyObject *o, long long *out) {
    if (!PyLong_Check(o)) {
        if (!PyIndex_Check(o)) return false;   // a NumPy integer
        PyObject *i = PyNumber_Index(o);
        if (!i) {
            PyErr_Clear();
            return false;
        }
        const bool ok = to_integer(i, out);
        Py_DECREF(i);
        return ok;
    }
    int overflow = 0;
    *out = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

template <typename T>
struct Arg {   // int, int64_t, size_t, uint32_t, int32_t
    static bool from(PyObject *o, T *out, Views &) {
        long long v;
        if (!to_integer(o, &v) || (long long)(T)v != v) return false;
        *out = (T)v;
        return true;
    }
};
template <>
struct Arg<float> {
    static bool from(PyObject *o, float *out, Views &) {
        if (!PyFloat_Check(o) && !PyLong_CheckExact(o)) return false;
        *out = (float)PyFloat_AsDouble(o);
        if (PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
        return true;
    }
};
template <typename T>
struct Arg<T *> {
    static bool from(PyObject *o, T **out, Views &views) {
        if (o == Py_None) {
            *out = nullptr;
            return true;
        }
        if (PyLong_CheckExact(o)) {
            const unsigned long long v = PyLong_AsUnsignedLongLong(o);
            if (v == (unsigned long long)-1 && PyErr_Occurred()) {
                PyErr_Clear();
                return false;
            }
            *out = reinterpret_cast<T *>((uintptr_t)v);
            return true;
        }
        const bool holder = Py_TYPE(o) == g_c_void_p;
        if (views.n >= 8 || !(holder || PyObject_TypeCheck(o, g_ndarray) || PyObject_TypeCheck(o, g_structure))) return false;
        Py_buffer *b = &views.held[views.n];
        constexpr bool floats = std::is_same_v<T, const float>;   // (an array behind a typed pointer has to hold that type)
        if (PyObject_GetBuffer(o, b, floats ? PyBUF_SIMPLE | PyBUF_FORMAT : PyBUF_SIMPLE) != 0) {
            PyErr_Clear();
            return false;
        }
        if (floats && !holder && !(b->format && strcmp(b->format, "f") == 0)) {
            PyBuffer_Release(b);
            return false;
        }
        if (holder) {   // the pointer it holds, not where it is held
            memcpy(out, b->buf, sizeof *out);
            PyBuffer_Release(b);
            return true;
        }
        views.n++;   // released after the call
        *out = static_cast<T *>(b->buf);
        return true;
    }
};

struct Call {
    PyObject_HEAD
    vectorcallfunc vector;
    void *address;
    PyObject *fallback;   // the ctypes function
};

template <typename F>
struct Binder;
template <typename... A>
struct Binder<int(A...)> {
    template <size_t... I>
    static PyObject *run(Call *self, PyObject *const *args, size_t nargsf, PyObject *kw, std::index_sequence<I...>) {
        const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
        Views views;
        std::tuple<A...> v;
        if (n != (Py_ssize_t)sizeof...(A) || kw || !(Arg<A>::from(args[I], &std::get<I>(v), views) && ...))
            return PyObject_Vectorcall(self->fallback, args, (size_t)n, kw);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = reinterpret_cast<int (*)(A...)>(self->address)(std::get<I>(v)...);
        Py_END_ALLOW_THREADS
        return PyLong_FromLong(rc);
    }
    static PyObject *call(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kw) {
        return run(reinterpret_cast<Call *>(self), args, nargsf, kw, std::index_sequence_for<A...>{});
    }
};

struct Entry {
    const char *name;
    vectorcallfunc call;
};
#define BIND(f) {#f, Binder<decltype(f)>::call}
const Entry kEntries[] = {
    BIND(hipc_fill), BIND(hipc_copy), BIND(hipc_graph_launch), BIND(hipc_matmul_nbits), BIND(hipc_matmul_nbits_packed),
    BIND(hipc_dynamic_quantize_linear), BIND(hipc_dynamic_quantize_linear_static), BIND(hipc_decomposed_gelu),
    BIND(hipc_dynamic_quantize_linear_gelu), BIND(hipc_matmul_integer), BIND(hipc_matmul_integer_raw),
    BIND(hipc_matmul_integer_scale_bias), BIND(hipc_requantize), BIND(hipc_qlinear_matmul), BIND(hipc_conv_integer),
    BIND(hipc_qlinear_conv), BIND(hipc_decoder_reset), BIND(hipc_decoder_step),
};
#undef BIND

void call_dealloc(PyObject *self) {
    Py_XDECREF(reinterpret_cast<Call *>(self)->fallback);
    Py_TYPE(self)->tp_free(self);
}
PyTypeObject CallType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// bind(name, address, ctypes function) -> a callable, or None where the name has no entry here
PyObject *bind(PyObject *, PyObject *args) {
    const char *name;
    unsigned long long address;
    PyObject *fallback;
    if (!PyArg_ParseTuple(args, "sKO", &name, &address, &fallback)) return nullptr;
    for (const Entry &e : kEntries)
        if (strcmp(e.name, name) == 0) {
            Call *c = PyObject_New(Call, &CallType);
            if (!c) return nullptr;
            c->vector = e.call, c->address = reinterpret_cast<void *>((uintptr_t)address), c->fallback = fallback;
            Py_INCREF(fallback);
            return reinterpret_cast<PyObject *>(c);
        }
    Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {{"bind", bind, METH_VARARGS, "bind(name, address, ctypes function) -> callable or None"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall(void) {
    CallType.tp_name = "onnx_vulkan_rs_amd._fastcall.Call";
    CallType.tp_basicsize = sizeof(Call);
    CallType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    CallType.tp_vectorcall_offset = offsetof(Call, vector);
    CallType.tp_call = PyVectorcall_Call;
    CallType.tp_dealloc = call_dealloc;
    if (PyType_Ready(&CallType) < 0) return nullptr;
    auto type_of = [](const char *module, const char *name) -> PyTypeObject * {
        PyObject *m = PyImport_ImportModule(module);
        PyObject *t = m ? PyObject_GetAttrString(m, name) : nullptr;
        Py_XDECREF(m);
        return reinterpret_cast<PyTypeObject *>(t);
    };
    if (!(g_c_void_p = type_of("ctypes", "c_void_p")) || !(g_structure = type_of("ctypes", "Structure")) || !(g_ndarray = type_of("numpy", "ndarray")))
        return nullptr;
    PyObject *m = PyModule_Create(&kModule);
    if (m && PyModule_AddStringConstant(m, "build_id", HIPC_BUILD_ID) < 0) Py_CLEAR(m);
    return m;
}
