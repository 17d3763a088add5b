/* crow_nest_amd._launch: the package's way into crow_hip_launch_dims_split and crow_hip_launch without ctypes.
 *
 * A decode step is hundreds of small launches from Python, and converting their arguments through ctypes - a structure for
 * the dimensions, an array for the values, eight converted arguments, two calls - took longer than the launch itself.  This
 * module takes the same arguments as plain integers and calls the two entry points of the library that ctypes has loaded
 * (their addresses are handed to bind(); nothing is linked).  One projection [512, 2048]: 8.3 us a call through ctypes, of
 * which the launch itself is about 2.5.
 *
 * Both functions return the library's error code; the caller turns it into its exception. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "../../include/crow_hip.h"
#include "../../include/crow_hip_bench.h"

#define MAX_VALS 32

static int (*dims_fn)(const char*, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, crow_dims*);
static int (*launch_fn)(crow_fn_t, uint32_t, uint32_t, uint32_t, uint32_t, const uint64_t*, uint32_t, void*);

static PyObject* py_bind(PyObject* self, PyObject* args) {
    unsigned long long d, l;
    (void)self;
    if (!PyArg_ParseTuple(args, "KK", &d, &l)) return NULL;
    dims_fn = (int (*)(const char*, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, crow_dims*))(uintptr_t)d;
    launch_fn = (int (*)(crow_fn_t, uint32_t, uint32_t, uint32_t, uint32_t, const uint64_t*, uint32_t, void*))(uintptr_t)l;
    Py_RETURN_NONE;
}

/* n integers (or what has __index__: numpy's) of args -> out; 0 and an exception set if one is not an integer of 64 bits */
static int unpack(PyObject* const* args, Py_ssize_t n, uint64_t* out) {
    for (Py_ssize_t i = 0; i < n; i++) {
        if (PyLong_CheckExact(args[i])) {
            out[i] = PyLong_AsUnsignedLongLong(args[i]);
        } else {
            PyObject* v = PyNumber_Index(args[i]);
            if (v == NULL) return 0;
            out[i] = PyLong_AsUnsignedLongLong(v);
            Py_DECREF(v);
        }
        if (out[i] == (uint64_t)-1 && PyErr_Occurred()) return 0;
    }
    return 1;
}

static PyObject* checked(Py_ssize_t n, Py_ssize_t least) {
    if (launch_fn == NULL || dims_fn == NULL) return PyErr_Format(PyExc_RuntimeError, "_launch: bind() has not been called");
    if (n < least || n > MAX_VALS) return PyErr_Format(PyExc_TypeError, "_launch: %zd arguments", n);
    return Py_None;
}

/* launch(name: bytes, function, rows, k_dim, z, *values): the library's dimensions for this problem, then the launch */
static PyObject* py_launch(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    uint64_t v[MAX_VALS];
    (void)self;
    if (checked(nargs, 5) == NULL) return NULL;
    const char* name = PyBytes_AsString(args[0]);
    if (name == NULL || !unpack(args + 1, nargs - 1, v)) return NULL;
    if ((v[1] | v[2] | v[3]) > 0xFFFFFFFFull) return PyErr_Format(PyExc_OverflowError, "_launch: dimensions are 32-bit words");
    int rc;
    crow_dims d;
    Py_BEGIN_ALLOW_THREADS
    rc = dims_fn(name, (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3], 0, 0, &d);
    if (rc == CROW_OK) rc = launch_fn((crow_fn_t)(uintptr_t)v[0], d.gx, d.gy, d.gz, d.bx, v + 4, (uint32_t)(nargs - 5), NULL);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

/* launch_at(function, gx, gy, gz, bx, *values) */
static PyObject* py_launch_at(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    uint64_t v[MAX_VALS];
    (void)self;
    if (checked(nargs, 5) == NULL || !unpack(args, nargs, v)) return NULL;
    if ((v[1] | v[2] | v[3] | v[4]) > 0xFFFFFFFFull) return PyErr_Format(PyExc_OverflowError, "_launch: dimensions are 32-bit words");
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = launch_fn((crow_fn_t)(uintptr_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3], (uint32_t)v[4], v + 5, (uint32_t)(nargs - 5), NULL);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

static PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, "bind(address of crow_hip_launch_dims_split, address of crow_hip_launch)"},
    {"launch", (PyCFunction)(void (*)(void))py_launch, METH_FASTCALL, "launch(name, function, rows, k_dim, z, *values) -> error code"},
    {"launch_at", (PyCFunction)(void (*)(void))py_launch_at, METH_FASTCALL, "launch_at(function, gx, gy, gz, bx, *values) -> error code"},
    {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", NULL, -1, methods, NULL, NULL, NULL, NULL};
PyMODINIT_FUNC PyInit__launch(void) { return PyModule_Create(&module); }
