/* CPython calls of the entry points that a linear or an activation quantizer makes per call.
 *
 * A ctypes call with two dozen arguments converts each through a Python-level argument type (1.3 us
 * of a one-row linear's 11 us, whose kernel takes 8); these take the same integers (None for a missing
 * pointer) through the vectorcall protocol and call the C function by its declared type (0.3 us). The
 * functions are handed in by address (bind) from the libmq.so that kitchen_amd._lib has loaded, so there
 * is one copy of the library and this module links to nothing. The GIL is released around the call, as
 * ctypes does.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "../../include/mq.h"

#define MAX_ARGS 32

/* The n arguments as integers; bit i of `pointers`: argument i is a pointer, which None leaves null (anywhere
 * else None is refused, as ctypes refuses it: as 0 it would be an empty call or a default). */
static int ints(const char* what, PyObject* const* args, Py_ssize_t n, Py_ssize_t want, uint32_t pointers, int64_t* out) {
    if (n != want) {
        PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", what, want, n);
        return 0;
    }
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (args[i] == Py_None) {
            if (!(pointers >> i & 1)) {
                PyErr_Format(PyExc_TypeError, "%s: argument %zd must be an integer, not None", what, i + 1);
                return 0;
            }
            out[i] = 0;
        } else {
            out[i] = (int64_t)PyLong_AsLongLong(args[i]);
            if (out[i] == -1 && PyErr_Occurred()) return 0;
        }
    }
    return 1;
}

#define P(i) ((void*)(intptr_t)v[i])
#define I(i) ((int)v[i])
#define L(i) (v[i])

#define B(i) (UINT32_C(1) << (i))

/* name, number of arguments, which of them are pointers, call expression over v[] */
#define ENTRY(name, count, pointers, expr)                                               \
    static __typeof__(&name) fn_##name;                                                  \
    static PyObject* py_##name(PyObject* self, PyObject* const* args, Py_ssize_t n) {    \
        int64_t v[MAX_ARGS];                                                             \
        int rc;                                                                          \
        (void)self;                                                                      \
        if (!fn_##name) {                                                                \
            PyErr_SetString(PyExc_RuntimeError, #name " is not bound");                  \
            return NULL;                                                                 \
        }                                                                                \
        if (!ints(#name, args, n, count, pointers, v)) return NULL;                      \
        Py_BEGIN_ALLOW_THREADS                                                           \
        rc = expr;                                                                       \
        Py_END_ALLOW_THREADS                                                             \
        return PyLong_FromLong(rc);                                                      \
    }

ENTRY(mq_rotquant, 12, B(0) | B(8) | B(10) | B(11),
      fn_mq_rotquant(P(0), I(1), L(2), L(3), L(4), I(5), I(6), I(7), P(8), L(9), P(10), P(11)))
ENTRY(mq_swiglu_rotquant, 13, B(0) | B(9) | B(11) | B(12),
      fn_mq_swiglu_rotquant(P(0), I(1), L(2), L(3), L(4), I(5), I(6), I(7), I(8), P(9), L(10), P(11), P(12)))
ENTRY(mq_linear_w4_group, 23, B(0) | B(6) | B(8) | B(10) | B(12) | B(14) | B(20) | B(22),
      fn_mq_linear_w4_group(P(0), I(1), L(2), I(3), I(4), I(5), P(6), L(7), P(8), L(9), P(10), L(11), P(12), I(13),
                            P(14), I(15), L(16), L(17), L(18), L(19), P(20), L(21), P(22)))
ENTRY(mq_linear_rowscale, 21, B(0) | B(6) | B(9) | B(10) | B(12) | B(18) | B(20),
      fn_mq_linear_rowscale(P(0), I(1), L(2), I(3), I(4), I(5), P(6), L(7), I(8), P(9), P(10), I(11), P(12), I(13),
                            L(14), L(15), L(16), L(17), P(18), L(19), P(20)))

/* bind(rotquant, swiglu_rotquant, linear_w4_group, linear_rowscale): the functions' addresses */
static PyObject* py_bind(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    int64_t v[MAX_ARGS];
    (void)self;
    if (!ints("bind", args, n, 4, 0, v)) return NULL;
    fn_mq_rotquant = (__typeof__(fn_mq_rotquant))P(0);
    fn_mq_swiglu_rotquant = (__typeof__(fn_mq_swiglu_rotquant))P(1);
    fn_mq_linear_w4_group = (__typeof__(fn_mq_linear_w4_group))P(2);
    fn_mq_linear_rowscale = (__typeof__(fn_mq_linear_rowscale))P(3);
    Py_RETURN_NONE;
}

#define METHOD(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {
    METHOD("bind", py_bind),
    METHOD("mq_rotquant", py_mq_rotquant),
    METHOD("mq_swiglu_rotquant", py_mq_swiglu_rotquant),
    METHOD("mq_linear_w4_group", py_mq_linear_w4_group),
    METHOD("mq_linear_rowscale", py_mq_linear_rowscale),
    {NULL, NULL, 0, NULL},
};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", NULL, -1, methods, NULL, NULL, NULL, NULL};

/* ABI_VERSION: of the header whose argument orders are compiled in above */
PyMODINIT_FUNC PyInit__fast(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddIntConstant(m, "ABI_VERSION", MQ_ABI_VERSION) < 0) Py_CLEAR(m);
    return m;
}
