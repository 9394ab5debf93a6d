// The launch entry points as a CPython function: a layer's run() reaches the library without ctypes and its conversion of five
// arguments.  A call takes the host 3.7 to 3.9 us this way and 3.9 to 4.1 through ctypes (2000 calls of a small layer in a row); that shows
// where the host is the limit (FullyConnected 64 -> 16: 3.8 against 4.0 us a call) and not where the device is (4096 -> 4096 at one
// row, three sets of weights in turn: 4.7 against 4.6).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>

namespace
{
typedef int (*RunFn)(void* plan, uint32_t batch, const void* input, void* output, void* stream);

bool Address(PyObject* o, void** p)
{
    if (o == Py_None) { *p = nullptr; return true; }
    if (!PyLong_CheckExact(o))
    {
        PyErr_SetString(PyExc_TypeError, "an address is an int or None");
        return false;
    }
    *p = reinterpret_cast<void*>(PyLong_AsUnsignedLongLongMask(o));      // (as ctypes converts: modulo 2^64)
    return true;
}

// run(function address, plan, batch, input, output, stream) -> status
PyObject* Run(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    void *fn, *plan, *input, *output, *stream;
    if (n != 6 || !PyLong_CheckExact(args[2]))
    {
        PyErr_SetString(PyExc_TypeError, "run(function, plan, batch, input, output, stream)");
        return nullptr;
    }
    if (!Address(args[0], &fn) || !Address(args[1], &plan) || !Address(args[3], &input) || !Address(args[4], &output) || !Address(args[5], &stream)) return nullptr;
    const uint32_t batch = static_cast<uint32_t>(PyLong_AsUnsignedLongMask(args[2]));
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = reinterpret_cast<RunFn>(fn)(plan, batch, input, output, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

PyMethodDef methods[] = {{"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Run)), METH_FASTCALL, "run(function, plan, batch, input, output, stream) -> status"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
} // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&module); }
