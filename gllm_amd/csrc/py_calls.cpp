// The C entry points that a model's step calls, as Python functions that take plain numbers.
//
// Through ctypes a call of eleven arguments takes 0.9 us of the 4.9 that the smallest matmul takes from Python; here the numbers are read
// straight out of the argument array.  What is accepted, and what an argument of another type raises, is as ctypes has it for these
// prototypes: whole numbers (their low bits), None for a null pointer.  The interpreter's lock is released around the call.
//
// The functions are bound to addresses in the library that is already loaded (bind(name, address)); this module links nothing of it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "gllm_hip_quant.h"

namespace {

PyObject *argument_error = nullptr; // ctypes.ArgumentError

bool refuse(Py_ssize_t i, const char *expected, PyObject *got)
{
    PyErr_Format(argument_error, "argument %zd: TypeError: %s expected instead of %s instance", i + 1, expected, Py_TYPE(got)->tp_name);
    return false;
}

template <class T>
bool read(PyObject *v, Py_ssize_t i, T &out)
{
    if constexpr (std::is_floating_point_v<T>) {
        const double d = PyFloat_AsDouble(v);
        if (d == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            return refuse(i, "float", v);
        }
        out = static_cast<T>(d);
        return true;
    } else {
        if (std::is_pointer_v<T> && v == Py_None) {
            out = T{};
            return true;
        }
        if (!PyLong_Check(v)) return refuse(i, "int", v);
        const unsigned long long bits = PyLong_AsUnsignedLongLongMask(v);
        if constexpr (std::is_pointer_v<T>) out = reinterpret_cast<T>(static_cast<uintptr_t>(bits));
        else out = static_cast<T>(bits);
        return true;
    }
}

template <class Fn> struct Call;
template <class... A>
struct Call<int(A...)> {
    template <size_t... I>
    static PyObject *run(PyObject *self, PyObject *const *args, std::index_sequence<I...>)
    {
        std::tuple<std::decay_t<A>...> t;
        if (!(read(args[I], static_cast<Py_ssize_t>(I), std::get<I>(t)) && ...)) return nullptr;
        auto fn = reinterpret_cast<int (*)(A...)>(PyCapsule_GetPointer(self, nullptr));
        if (!fn) return nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = fn(std::get<I>(t)...);
        Py_END_ALLOW_THREADS
        return PyLong_FromLong(rc);
    }
    static PyObject *invoke(PyObject *self, PyObject *const *args, Py_ssize_t n)
    {
        if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
            PyErr_Format(PyExc_TypeError, "this function takes %zd arguments (%zd given)", static_cast<Py_ssize_t>(sizeof...(A)), n);
            return nullptr;
        }
        return run(self, args, std::index_sequence_for<A...>{});
    }
};

#define GLLMQ_CALL(NAME) { #NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Call<decltype(NAME)>::invoke)), METH_FASTCALL, nullptr }
PyMethodDef calls[] = {
    GLLMQ_CALL(gllmq_quantized_matmul_ex), GLLMQ_CALL(gllmq_quantized_matmul_elem), GLLMQ_CALL(gllmq_quantized_matmul_batch),
    GLLMQ_CALL(gllmq_dequantize), GLLMQ_CALL(gllmq_quant_gather), GLLMQ_CALL(gllmq_quant_gather_elem),
    GLLMQ_CALL(gllmq_ffn_swiglu), GLLMQ_CALL(gllmq_ffn_swiglu_elem), GLLMQ_CALL(gllmq_argmax), GLLMQ_CALL(gllmq_lm_head_argmax),
    GLLMQ_CALL(gllmq_moe_route), GLLMQ_CALL(gllmq_moe_matvec), GLLMQ_CALL(gllmq_moe_matvec_elem),
};

PyObject *bind(PyObject *, PyObject *args)
{
    const char *name;
    unsigned long long address;
    if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
    for (PyMethodDef &c : calls)
        if (std::strcmp(c.ml_name, name) == 0) {
            PyObject *at = PyCapsule_New(reinterpret_cast<void *>(static_cast<uintptr_t>(address)), nullptr, nullptr);
            if (!at) return nullptr;
            PyObject *fn = PyCFunction_New(&c, at);
            Py_DECREF(at);
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
    PyObject *ctypes = PyImport_ImportModule("ctypes");
    if (!ctypes) return nullptr;
    argument_error = PyObject_GetAttrString(ctypes, "ArgumentError");
    Py_DECREF(ctypes);
    if (!argument_error) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (!m) return nullptr;
    PyObject *names = PyList_New(0);
    for (PyMethodDef &c : calls) {
        PyObject *s = names ? PyUnicode_FromString(c.ml_name) : nullptr;
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
