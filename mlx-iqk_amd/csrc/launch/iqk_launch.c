/* A CPython binding of the decode, verify and prefill entry points of
 * libiqk_hip.so: the launch paths an eager call of the switch module takes (a
 * 1-token dispatch's kernel runs for ~6 us, and a ctypes call with twelve
 * converted arguments costs ~4 us of host time).  Each function takes the C ABI's arguments as Python integers
 * (device pointers as addresses, the stream as its handle) and returns the
 * entry point's code; nothing else is done here.  It is built against the
 * library's own header and carries the digest of the sources it was built
 * with, which the loader compares with the library's. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <limits.h>
#include <stdint.h>

#include "iqk_hip.h"

#ifndef IQK_SOURCE_HASH
#define IQK_SOURCE_HASH "unset"
#endif

static int as_i64(PyObject *o, long long *v) {
    *v = PyLong_AsLongLong(o);
    return !(*v == -1 && PyErr_Occurred());
}

/* gemv(kind, member, n, out, num_experts, x, streams, n_streams, sel,
 *      pairs_per_row, mats, y, stream): kind 0 iqk_gemv, 1 iqk_gemv_floor,
 * 2 iqk_gemv_floor_grid, 3 iqk_gemv_ids64; streams is the address of the stream pointer array. */
static PyObject *gemv(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
    (void)self;
    if (nargs != 13) {
        PyErr_SetString(PyExc_TypeError, "gemv takes 13 integer arguments");
        return NULL;
    }
    long long v[13];
    for (int i = 0; i < 13; ++i)
        if (!as_i64(args[i], &v[i])) return NULL;
    /* the narrow arguments: member and stream count (int), pairs per row and
     * pair count (uint32); a value out of range is refused, not truncated */
    if (v[1] < INT_MIN || v[1] > INT_MAX || v[7] < INT_MIN || v[7] > INT_MAX || v[9] < 0 || v[9] > UINT32_MAX ||
        v[10] < 0 || v[10] > UINT32_MAX) {
        PyErr_SetString(PyExc_OverflowError, "gemv: member, stream count, pairs per row or pair count out of range");
        return NULL;
    }
    if (v[0] == 3) {
        const int rc = iqk_gemv_ids64((int)v[1], (int64_t)v[2], (int64_t)v[3], (int64_t)v[4],
                                      (const void *)(uintptr_t)v[5], (const void *const *)(uintptr_t)v[6], (int)v[7],
                                      (const int64_t *)(uintptr_t)v[8], (uint32_t)v[9], (uint32_t)v[10],
                                      (void *)(uintptr_t)v[11], (void *)(uintptr_t)v[12]);
        return PyLong_FromLong(rc);
    }
    int (*fn)(int, int64_t, int64_t, int64_t, const void *, const void *const *, int, const uint32_t *, uint32_t,
              uint32_t, void *, void *) = v[0] == 1 ? iqk_gemv_floor : v[0] == 2 ? iqk_gemv_floor_grid : iqk_gemv;
    const int rc = fn((int)v[1], (int64_t)v[2], (int64_t)v[3], (int64_t)v[4], (const void *)(uintptr_t)v[5],
                      (const void *const *)(uintptr_t)v[6], (int)v[7], (const uint32_t *)(uintptr_t)v[8],
                      (uint32_t)v[9], (uint32_t)v[10], (void *)(uintptr_t)v[11], (void *)(uintptr_t)v[12]);
    return PyLong_FromLong(rc);
}

static PyObject *refuse(const char *what) {
    PyErr_SetString(PyExc_OverflowError, what);
    return NULL;
}

/* sorted(union, member, n, out, num_experts, x, n_x_rows, streams, n_streams,
 *        sorted_ids, toks, mats, y, stream): iqk_gemv_sorted, or iqk_gemv_union. */
static PyObject *sorted(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
    (void)self;
    if (nargs != 14) {
        PyErr_SetString(PyExc_TypeError, "sorted takes 14 integer arguments");
        return NULL;
    }
    long long v[14];
    for (int i = 0; i < 14; ++i)
        if (!as_i64(args[i], &v[i])) return NULL;
    if (v[1] < INT_MIN || v[1] > INT_MAX || v[8] < INT_MIN || v[8] > INT_MAX || v[11] < 0 || v[11] > UINT32_MAX)
        return refuse("sorted: member, stream count or pair count out of range");
    const int rc = (v[0] ? iqk_gemv_union : iqk_gemv_sorted)(
        (int)v[1], (int64_t)v[2], (int64_t)v[3], (int64_t)v[4], (const void *)(uintptr_t)v[5], (int64_t)v[6],
        (const void *const *)(uintptr_t)v[7], (int)v[8], (const uint32_t *)(uintptr_t)v[9],
        (const uint32_t *)(uintptr_t)v[10], (uint32_t)v[11], (void *)(uintptr_t)v[12], (void *)(uintptr_t)v[13]);
    return PyLong_FromLong(rc);
}

/* prefill(member, n, out, num_experts, x, n_x_rows, streams, n_streams,
 *         row_start, rows, ids, wide, n_pairs, rows_per_pair, pairs_per_x_row,
 *         work, y, stream): iqk_prefill. */
static PyObject *prefill(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
    (void)self;
    if (nargs != 18) {
        PyErr_SetString(PyExc_TypeError, "prefill takes 18 integer arguments");
        return NULL;
    }
    long long v[18];
    for (int i = 0; i < 18; ++i)
        if (!as_i64(args[i], &v[i])) return NULL;
    if (v[0] < INT_MIN || v[0] > INT_MAX || v[7] < INT_MIN || v[7] > INT_MAX)
        return refuse("prefill: member or stream count out of range");
    const int rc = iqk_prefill((int)v[0], (int64_t)v[1], (int64_t)v[2], (int64_t)v[3], (const void *)(uintptr_t)v[4],
                               (int64_t)v[5], (const void *const *)(uintptr_t)v[6], (int)v[7], (int64_t)v[8],
                               (int64_t)v[9], (const void *)(uintptr_t)v[10], v[11] != 0, (int64_t)v[12],
                               (int64_t)v[13], (int64_t)v[14], (uint32_t *)(uintptr_t)v[15],
                               (void *)(uintptr_t)v[16], (void *)(uintptr_t)v[17]);
    return PyLong_FromLong(rc);
}

static PyObject *source_hash(PyObject *self, PyObject *unused) {
    (void)self;
    (void)unused;
    return PyUnicode_FromString(IQK_SOURCE_HASH);
}

static PyMethodDef methods[] = {
    {"gemv", (PyCFunction)(void (*)(void))gemv, METH_FASTCALL, "iqk_gemv / _floor / _floor_grid / _ids64"},
    {"sorted", (PyCFunction)(void (*)(void))sorted, METH_FASTCALL, "iqk_gemv_sorted / _union"},
    {"prefill", (PyCFunction)(void (*)(void))prefill, METH_FASTCALL, "iqk_prefill"},
    {"source_hash", source_hash, METH_NOARGS, "digest of the kernel sources this binding was built with"},
    {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_iqk_launch", NULL, -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__iqk_launch(void) { return PyModule_Create(&module); }
