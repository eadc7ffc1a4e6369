// Calls of the libraries' entry points from Python: bind(address, kinds) -> a function of as many arguments, which returns the status.
//
// kinds: a character for each argument, 'p' an address (None: null), 'i' a whole number, 'f' a float; at most 18 of the first two and two
// floats.  Under the x86-64 calling convention floats are passed apart from the others and a callee takes the lower bits of a wider argument, so
// that one call fits every such signature, as long as each argument is what the signature has in its place: a number of another kind would move
// those behind it.  ctypes converts each argument through an object of its own: nine arguments 2.3 us, fifteen 3.5; here 0.5.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <string.h>

#if !defined(__x86_64__)
#error "one call for all signatures rests on the x86-64 calling convention"
#endif

namespace {

constexpr Py_ssize_t kWhole = 18, kFloats = 2;
typedef uint64_t u;
typedef int (*Entry)(u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, u, float, float);

// An entry point, as the bytes that are the `self` of its function.
struct Bound {
    u address;
    Py_ssize_t count;
    char kinds[kWhole + kFloats];
};

PyObject* argument_error = nullptr;        // ctypes.ArgumentError

PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t count) {
    const Bound* b = (const Bound*)PyBytes_AS_STRING(self);
    if (count != b->count) return PyErr_Format(PyExc_TypeError, "this function takes %zd arguments (%zd given)", b->count, count);
    u v[kWhole] = {0};
    float f[kFloats] = {0.f, 0.f};
    Py_ssize_t whole = 0, floats = 0;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* a = args[i];
        if (b->kinds[i] == 'f') {
            const double d = PyFloat_AsDouble(a);
            if (d == -1. && PyErr_Occurred()) return PyErr_Format(argument_error, "argument %zd: a float is expected, not %s", i + 1, Py_TYPE(a)->tp_name);
            f[floats++] = (float)d;
        } else if (a == Py_None && b->kinds[i] == 'p') {
            v[whole++] = 0;
        } else {
            // as ctypes: what has an index is a whole number, a float is none
            const u n = PyFloat_Check(a) ? (u)-1 : PyLong_AsUnsignedLongLongMask(a);
            if (n == (u)-1 && (PyFloat_Check(a) || PyErr_Occurred()))
                return PyErr_Format(argument_error, "argument %zd: a whole number is expected, not %s", i + 1, Py_TYPE(a)->tp_name);
            v[whole++] = n;
        }
    }
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = ((Entry)b->address)(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11], v[12], v[13], v[14], v[15], v[16], v[17],
                                 f[0], f[1]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

PyMethodDef entry = {"entry", (PyCFunction)(void (*)(void))call, METH_FASTCALL, "an entry point of a library: status"};

PyObject* bind(PyObject*, PyObject* args) {
    unsigned long long address;
    const char* kinds;
    if (!PyArg_ParseTuple(args, "Ks", &address, &kinds)) return nullptr;
    Bound b;
    memset(&b, 0, sizeof(b));
    b.address = address;
    b.count = (Py_ssize_t)strlen(kinds);
    Py_ssize_t floats = 0;
    for (Py_ssize_t i = 0; i < b.count; ++i) floats += kinds[i] == 'f';
    if (address == 0 || strspn(kinds, "pif") != (size_t)b.count || floats > kFloats || b.count - floats > kWhole)
        return PyErr_Format(PyExc_ValueError, "no entry point, or one of other arguments than %zd addresses and whole numbers and %zd floats", kWhole, kFloats);
    memcpy(b.kinds, kinds, (size_t)b.count);
    PyObject* self = PyBytes_FromStringAndSize((const char*)&b, sizeof(b));
    if (!self) return nullptr;
    PyObject* f = PyCFunction_New(&entry, self);
    Py_DECREF(self);
    return f;
}

PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, "bind(address, kinds) -> function of an entry point"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call(void) {
    PyObject* ctypes = PyImport_ImportModule("ctypes");
    if (!ctypes) return nullptr;
    argument_error = PyObject_GetAttrString(ctypes, "ArgumentError");
    Py_DECREF(ctypes);
    return argument_error ? PyModule_Create(&module) : nullptr;
}
