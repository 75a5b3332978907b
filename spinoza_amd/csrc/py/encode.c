/*
 * encode.c -- op dicts to the C ABI's spz_op records (CPython extension
 * spinoza_amd._encode, used by executor.encode_ops).
 *
 * Filling ctypes structures field by field costs about 0.43 us per op, 16 ms
 * for the 36746 ops of a 128-circuit batch, a third of the whole call; here an
 * op is ten dict lookups and stores.  Conversions are those of int(), float()
 * and bool() on the dict's values; integers that do not fit wrap as ctypes
 * assignments do.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <string.h>

#include "../../../include/spinoza_amd.h"

enum { F_KIND, F_TARGET, F_THETA, F_PHI, F_LAM, F_T1, F_CLASSICAL, F_ONES, F_ZEROS, F_U, F_MATRIX,
       F_COUNT };
static const char *const names[F_COUNT] = {"kind", "target", "theta", "phi", "lam", "t1",
                                           "classical", "ones", "zeros", "u", "matrix"};
static PyObject *keys[F_COUNT];

/* Borrowed value of a field, NULL without an error when it is absent. */
static PyObject *field(PyObject *d, int f) { return PyDict_GetItemWithError(d, keys[f]); }

static int as_bits(PyObject *v, uint64_t *out)
{
    if (PyLong_CheckExact(v)) {
        *out = PyLong_AsUnsignedLongLongMask(v);
    } else {
        PyObject *n = PyNumber_Long(v);
        if (!n) return -1;
        *out = PyLong_AsUnsignedLongLongMask(n);
        Py_DECREF(n);
    }
    return PyErr_Occurred() ? -1 : 0;
}

static int as_real(PyObject *v, double *out)
{
    if (PyFloat_CheckExact(v)) {
        *out = PyFloat_AS_DOUBLE(v);
        return 0;
    }
    PyObject *n = PyNumber_Float(v);
    if (!n) return -1;
    *out = PyFloat_AS_DOUBLE(n);
    Py_DECREF(n);
    return 0;
}

static int get_bits(PyObject *d, int f, uint64_t *out)
{
    PyObject *v = field(d, f);
    if (!v) return PyErr_Occurred() ? -1 : 0;
    return as_bits(v, out);
}

static int get_real(PyObject *d, int f, double *out)
{
    PyObject *v = field(d, f);
    if (!v) return PyErr_Occurred() ? -1 : 0;
    return as_real(v, out);
}

static int one(PyObject *d, spz_op *o, int *has_matrix)
{
    uint64_t kind = 0, target = 0, t1 = 0, ones = 0, zeros = 0;
    double theta = 0.0, phi = 0.0, lam = 0.0, u = 1.0;
    PyObject *k = field(d, F_KIND);
    if (!k) {
        if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, keys[F_KIND]);
        return -1;
    }
    if (as_bits(k, &kind) || get_bits(d, F_TARGET, &target) || get_real(d, F_THETA, &theta) ||
        get_real(d, F_PHI, &phi) || get_real(d, F_LAM, &lam) || get_bits(d, F_T1, &t1) ||
        get_bits(d, F_ONES, &ones) || get_bits(d, F_ZEROS, &zeros) || get_real(d, F_U, &u))
        return -1;
    int classical = 0;
    PyObject *c = field(d, F_CLASSICAL);
    if (c) classical = PyObject_IsTrue(c);
    if (classical < 0 || PyErr_Occurred()) return -1;
    memset(o, 0, sizeof *o);
    o->kind = (int32_t)(uint32_t)kind;
    o->target = (int32_t)(uint32_t)target;
    o->theta = theta;
    o->phi = phi;
    o->lambda = lam;
    o->t1 = (int32_t)(uint32_t)t1;
    o->flags = classical ? SPZ_OPF_CLASSICAL : 0;
    o->ones = ones;
    o->zeros = zeros;
    o->u = u;
    *has_matrix = field(d, F_MATRIX) != NULL;
    return PyErr_Occurred() ? -1 : 0;
}

/* fill(ops, buffer) -> indices of the ops that carry a matrix.  `ops` is a
 * sequence of dicts, `buffer` a writable buffer of len(ops) spz_op. */
static PyObject *fill(PyObject *self, PyObject *args)
{
    PyObject *ops;
    Py_buffer buf;
    (void)self;
    if (!PyArg_ParseTuple(args, "Ow*", &ops, &buf)) return NULL;
    PyObject *found = NULL, *seq = PySequence_Fast(ops, "ops must be a sequence of dicts");
    if (!seq) goto done;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
    if ((size_t)buf.len / sizeof(spz_op) < (size_t)n) {
        PyErr_SetString(PyExc_ValueError, "buffer too small for the ops");
        goto done;
    }
    found = PyList_New(0);
    for (Py_ssize_t i = 0; found && i < n; i++) {
        PyObject *d = PySequence_Fast_GET_ITEM(seq, i);
        int has_matrix = 0;
        int bad;
        if (PyDict_Check(d)) {
            bad = one(d, (spz_op *)buf.buf + i, &has_matrix);
        } else { /* another mapping */
            PyObject *copy = PyDict_New();
            bad = !copy || PyDict_Update(copy, d);
            if (bad && PyErr_ExceptionMatches(PyExc_AttributeError))
                PyErr_SetString(PyExc_TypeError, "an op is a mapping of its fields");
            bad = bad || one(copy, (spz_op *)buf.buf + i, &has_matrix);
            Py_XDECREF(copy);
        }
        if (bad) {
            Py_CLEAR(found);
        } else if (has_matrix) {
            PyObject *idx = PyLong_FromSsize_t(i);
            if (!idx || PyList_Append(found, idx)) Py_CLEAR(found);
            Py_XDECREF(idx);
        }
    }
done:
    Py_XDECREF(seq);
    PyBuffer_Release(&buf);
    return found;
}

static PyMethodDef methods[] = {
    {"fill", fill, METH_VARARGS, "fill(ops, buffer): encode op dicts as spz_op records"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_encode", NULL, -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__encode(void)
{
    for (int f = 0; f < F_COUNT; f++) {
        keys[f] = PyUnicode_InternFromString(names[f]);
        if (!keys[f]) return NULL;
    }
    return PyModule_Create(&module);
}
