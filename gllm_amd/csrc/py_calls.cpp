// The C entry points that a model's step calls, as Python functions that take plain numbers.
//
// Through ctypes a call of eleven arguments takes 0.9 us of the 4.9 that the smallest matmul takes from Python; here the numbers are read
// straight out of the argument array.  That is for int, float and None as the caller of every step has them; a call with anything else
// (an integer of numpy's, a ctypes object, a wrong type) goes through ctypes, which accepts and refuses what it does for these
// prototypes.  The interpreter's lock is released around the call.
//
// The functions are bound to addresses in the library that is already loaded (bind(name, address)); this module links nothing of it.
// It keeps to Python's limited interface, so that interpreters from 3.10 on load one build of it.
#define PY_SSIZE_T_CLEAN
#define Py_LIMITED_API 0x030A0000
#include <Python.h>

#include <cstdint>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "gllm_hip_quant.h"

namespace {

// False, without an exception: not a plain number of the kind.
template <class T>
bool read(PyObject *v, T &out)
{
    if constexpr (std::is_floating_point_v<T>) {
        if (!PyFloat_CheckExact(v)) return false;
        out = static_cast<T>(PyFloat_AsDouble(v));
        return true;
    } else {
        if (std::is_pointer_v<T> && v == Py_None) {
            out = T{};
            return true;
        }
        if (!PyLong_CheckExact(v) && !PyBool_Check(v)) return false;
        const unsigned long long bits = PyLong_AsUnsignedLongLongMask(v); // (the low bits, as ctypes takes them)
        if constexpr (std::is_pointer_v<T>) out = reinterpret_cast<T>(static_cast<uintptr_t>(bits));
        else out = static_cast<T>(bits);
        return true;
    }
}

template <class T>
const char *ctypes_name()
{
    if (std::is_pointer_v<T>) return "c_void_p";
    if (std::is_same_v<T, float>) return "c_float";
    if (std::is_same_v<T, uint32_t>) return "c_uint32";
    if (std::is_same_v<T, int>) return "c_int";
    static_assert(std::is_pointer_v<T> || std::is_same_v<T, float> || std::is_same_v<T, uint32_t> || std::is_same_v<T, int> || std::is_same_v<T, size_t>, "a type without a name here");
    return "c_size_t";
}

// self: a capsule of the C function's address, its context the same function through ctypes
template <class Fn> struct Call;
template <class... A>
struct Call<int(A...)> {
    template <size_t... I>
    static PyObject *run(PyObject *self, PyObject *const *args, Py_ssize_t n, std::index_sequence<I...>)
    {
        if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
            PyErr_Format(PyExc_TypeError, "this function takes %zd arguments (%zd given)", static_cast<Py_ssize_t>(sizeof...(A)), n);
            return nullptr;
        }
        std::tuple<std::decay_t<A>...> t;
        if (!(read(args[I], std::get<I>(t)) && ...)) return through_ctypes(self, args, n);
        auto fn = reinterpret_cast<int (*)(A...)>(PyCapsule_GetPointer(self, nullptr));
        if (!fn) return nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = fn(std::get<I>(t)...);
        Py_END_ALLOW_THREADS
        return PyLong_FromLong(rc);
    }
    static PyObject *through_ctypes(PyObject *self, PyObject *const *args, Py_ssize_t n)
    {
        PyObject *fn = static_cast<PyObject *>(PyCapsule_GetContext(self)), *all = fn ? PyTuple_New(n) : nullptr;
        if (!all) return nullptr;
        for (Py_ssize_t i = 0; i < n; ++i) {
            Py_INCREF(args[i]);
            PyTuple_SetItem(all, i, args[i]);
        }
        PyObject *rc = PyObject_CallObject(fn, all);
        Py_DECREF(all);
        return rc;
    }
    static PyObject *invoke(PyObject *self, PyObject *const *args, Py_ssize_t n) { return run(self, args, n, std::index_sequence_for<A...>{}); }
    // ctypes.CFUNCTYPE(c_int, types of the arguments)(address)
    static PyObject *ctypes_function(unsigned long long address)
    {
        PyObject *ctypes = PyImport_ImportModule("ctypes"), *fn = nullptr;
        if (!ctypes) return nullptr;
        const char *const names[] = { "c_int", ctypes_name<std::decay_t<A>>()... };
        PyObject *types = PyTuple_New(1 + sizeof...(A));
        for (size_t i = 0; types && i < 1 + sizeof...(A); ++i) {
            PyObject *type = PyObject_GetAttrString(ctypes, names[i]);
            if (!type || PyTuple_SetItem(types, static_cast<Py_ssize_t>(i), type) != 0) {
                Py_DECREF(types);
                types = nullptr;
            }
        }
        PyObject *make = types ? PyObject_GetAttrString(ctypes, "CFUNCTYPE") : nullptr, *prototype = make ? PyObject_CallObject(make, types) : nullptr;
        if (prototype) fn = PyObject_CallFunction(prototype, "K", address);
        Py_XDECREF(prototype);
        Py_XDECREF(make);
        Py_XDECREF(types);
        Py_DECREF(ctypes);
        return fn;
    }
};

struct Entry {
    PyMethodDef method;
    PyObject *(*ctypes_function)(unsigned long long);
};
#define GLLMQ_CALL(NAME)                                                                                                                             \
    { { #NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Call<decltype(NAME)>::invoke)), METH_FASTCALL, nullptr }, \
      &Call<decltype(NAME)>::ctypes_function }
Entry calls[] = {
    GLLMQ_CALL(gllmq_quantized_matmul_ex), GLLMQ_CALL(gllmq_quantized_matmul_elem), GLLMQ_CALL(gllmq_quantized_matmul_batch),
    GLLMQ_CALL(gllmq_dequantize), GLLMQ_CALL(gllmq_quant_gather), GLLMQ_CALL(gllmq_quant_gather_elem),
    GLLMQ_CALL(gllmq_ffn_swiglu), GLLMQ_CALL(gllmq_ffn_swiglu_elem), GLLMQ_CALL(gllmq_argmax), GLLMQ_CALL(gllmq_lm_head_argmax),
    GLLMQ_CALL(gllmq_moe_route), GLLMQ_CALL(gllmq_moe_matvec), GLLMQ_CALL(gllmq_moe_matvec_elem),
};

void release(PyObject *capsule) { Py_XDECREF(static_cast<PyObject *>(PyCapsule_GetContext(capsule))); }

PyObject *bind(PyObject *, PyObject *args)
{
    const char *name;
    unsigned long long address;
    if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
    for (Entry &c : calls)
        if (std::strcmp(c.method.ml_name, name) == 0) {
            PyObject *slow = c.ctypes_function(address);
            if (!slow) return nullptr;
            PyObject *at = PyCapsule_New(reinterpret_cast<void *>(static_cast<uintptr_t>(address)), nullptr, release), *fn = nullptr;
            if (at && PyCapsule_SetContext(at, slow) == 0) fn = PyCFunction_New(&c.method, at);
            else Py_DECREF(slow);
            Py_XDECREF(at);
            return fn;
        }
    PyErr_Format(PyExc_KeyError, "%s", name);
    return nullptr;
}

PyMethodDef methods[] = {
    { "bind", bind, METH_VARARGS, "bind(name, address): the C function at that address, called with plain numbers" },
    { nullptr, nullptr, 0, nullptr },
};
PyModuleDef module = { PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr };

} // namespace

PyMODINIT_FUNC PyInit__calls()
{
    PyObject *m = PyModule_Create(&module);
    if (!m) return nullptr;
    PyObject *names = PyList_New(0);
    for (const Entry &c : calls) {
        PyObject *s = names ? PyUnicode_FromString(c.method.ml_name) : nullptr;
        if (!s || PyList_Append(names, s) != 0) {
            Py_XDECREF(s);
            Py_XDECREF(names);
            Py_DECREF(m);
            return nullptr;
        }
        Py_DECREF(s);
    }
    if (PyModule_AddObject(m, "names", names) != 0) {
        Py_DECREF(names);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
