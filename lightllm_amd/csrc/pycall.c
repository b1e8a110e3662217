/* CPython entry of the one-call linear.  ctypes converts the eighteen arguments of mi355_block_fp8_linear in about 1.7 us, a
 * fifth of what a small decode linear costs on the host and more than its kernel's launch; taken from the argument vector
 * they are a quarter of a microsecond.  The call itself is the C entry of libmi355fp8.so, without the interpreter lock, as
 * ctypes makes it.  The entry's address comes from the library that the package has loaded: this file links against nothing,
 * so that a package that was copied or moved calls its own library. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "../../include/mi355_fp8.h"

enum { kArgs = 18 };

typedef __typeof__(&mi355_block_fp8_linear) linear_entry;

/* linear(x, x_dtype, W, Ws, C, M, N, K, ldw, ws_n, ws_k, ldc, x_q, x_s, ws, ws_bytes, c_dtype, stream) -> status.  Integers;
 * None is a null pointer.  `self` is the capsule of the C entry. */
static PyObject *linear(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
    const linear_entry entry = (linear_entry)(uintptr_t)PyCapsule_GetPointer(self, NULL);
    if (!entry) return NULL;
    if (nargs != kArgs) {
        PyErr_Format(PyExc_TypeError, "linear takes %d arguments (%zd given)", (int)kArgs, nargs);
        return NULL;
    }
    uint64_t v[kArgs];
    for (int i = 0; i < kArgs; ++i) {
        if (args[i] == Py_None) {
            v[i] = 0;
            continue;
        }
        if (!PyLong_Check(args[i])) {
            PyErr_Format(PyExc_TypeError, "argument %d of linear is not an integer", i + 1);
            return NULL;
        }
        const int64_t s = PyLong_AsLongLong(args[i]);
        if (s == -1 && PyErr_Occurred()) {
            PyErr_Clear(); /* an address in the upper half */
            v[i] = PyLong_AsUnsignedLongLong(args[i]);
            if (PyErr_Occurred()) return NULL;
        } else {
            v[i] = (uint64_t)s;
        }
    }
    int code;
    Py_BEGIN_ALLOW_THREADS
    code = entry((const void *)v[0], (int32_t)v[1], (const void *)v[2], (const float *)v[3], (void *)v[4], (int64_t)v[5],
                 (int64_t)v[6], (int64_t)v[7], (int64_t)v[8], (int64_t)v[9], (int64_t)v[10], (int64_t)v[11], (void *)v[12],
                 (float *)v[13], (void *)v[14], (size_t)v[15], (int32_t)v[16], (void *)v[17]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(code);
}

static PyMethodDef linear_method = {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL,
                                    "mi355_block_fp8_linear over integers"};

/* linear_at(address of mi355_block_fp8_linear) -> linear */
static PyObject *linear_at(PyObject *self, PyObject *address) {
    (void)self;
    void *entry = PyLong_AsVoidPtr(address);
    if (!entry) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "the address of the entry is null");
        return NULL;
    }
    PyObject *capsule = PyCapsule_New(entry, NULL, NULL);
    if (!capsule) return NULL;
    PyObject *call = PyCFunction_New(&linear_method, capsule);
    Py_DECREF(capsule);
    return call;
}

static PyMethodDef methods[] = {
    {"linear_at", linear_at, METH_O, "the one-call linear at the address of its C entry"},
    {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mi355call", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__mi355call(void) { return PyModule_Create(&module); }
