// Calls of the libraries' entry points from Python: call(address, arguments ...) -> status.
//
// Whole numbers and addresses (None: null) as 64-bit arguments, floats as floats; an entry point takes at most 18 of the former and
// two of the latter.  Under the x86-64 calling convention the two kinds are passed apart and a callee takes the lower bits of a wider
// argument, so that one call fits every such signature.  ctypes converts each argument through an object of its own: nine
// arguments 2.3 us, fifteen 3.5; here 0.5.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#if !defined(__x86_64__)
#error "one call for all signatures rests on the x86-64 calling convention"
#endif

namespace {

constexpr Py_ssize_t kWhole = 18, kFloats = 2;
typedef uint64_t u;
typedef int (*Entry)(u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, float, float);

PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t count) {
    u v[kWhole] = {0};
    float f[kFloats] = {0.f, 0.f};
    Py_ssize_t whole = 0, floats = 0;
    if (count < 1) return PyErr_Format(PyExc_TypeError, "an address is missing");
    const u address = PyLong_AsUnsignedLongLong(args[0]);
    if (PyErr_Occurred()) return nullptr;
    if (address == 0) return PyErr_Format(PyExc_ValueError, "null address");
    for (Py_ssize_t i = 1; i < count; ++i) {
        PyObject* a = args[i];
        if (PyFloat_Check(a)) {
            if (floats == kFloats) return PyErr_Format(PyExc_TypeError, "more than %d floats", (int)kFloats);
            f[floats++] = (float)PyFloat_AS_DOUBLE(a);
            continue;
        }
        if (whole == kWhole) return PyErr_Format(PyExc_TypeError, "more than %d whole numbers", (int)kWhole);
        v[whole++] = a == Py_None ? 0 : PyLong_AsUnsignedLongLongMask(a);
        if (v[whole - 1] == (u)-1 && PyErr_Occurred()) return nullptr;
    }
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = ((Entry)address)(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11], v[12], v[13], v[14], v[15], v[16], v[17],
                              f[0], f[1]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

PyMethodDef methods[] = {{"call", (PyCFunction)(void (*)(void))call, METH_FASTCALL, "call(address, arguments ...) -> status"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call(void) { return PyModule_Create(&module); }
