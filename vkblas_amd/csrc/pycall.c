/*
 * pycall.c — the Python binding's GEMM call without ctypes (module
 * vkblas_amd._call).
 *
 * A small GEMM is bound by its launch on the host, and ctypes' conversion of
 * 25 arguments was the largest part of that: 3.1 us for vkblas_gemm_async and
 * 3.7 for vkblas_gemm_ex_async with its structure, of about 8 a call.  Here
 * the arguments are read from the interpreter's vector directly.
 *
 * Arguments are converted as the ctypes prototypes of vkblas_amd/__init__.py
 * do: integers modulo 2^32 or 2^64, pointers from an int or None, floats from a
 * float or an int.  Anything else (a ctypes object, a subclass) returns None
 * and the caller makes the call through ctypes, whose rules then apply.  The
 * GIL is released during the call, as ctypes releases it.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include "vkblas_ext.h"

typedef vkblas_status_t (*gemm_ex_fn)(vkblas_dtype_t, vkblas_dtype_t, vkblas_op_t, vkblas_op_t, uint32_t, uint32_t,
                                      uint32_t, float, const void*, uint32_t, const void*, uint32_t, float, void*,
                                      uint32_t, uint32_t, int64_t, int64_t, int64_t, vkblas_scalar_mode_t,
                                      const void*, const void*, uint32_t, const vkblas_epilogue_t*, void*);

/* 1 and *v, or 0: not a plain int */
static int get_int(PyObject* o, unsigned long long* v) {
    if (!PyLong_CheckExact(o)) return 0;
    *v = PyLong_AsUnsignedLongLongMask(o);
    return !(*v == (unsigned long long)-1 && PyErr_Occurred());
}
static int get_ptr(PyObject* o, unsigned long long* v) {
    *v = 0;
    return o == Py_None || get_int(o, v);
}
static int get_float(PyObject* o, float* v) {
    if (PyFloat_CheckExact(o)) {
        *v = (float)PyFloat_AS_DOUBLE(o);
        return 1;
    }
    if (!PyLong_CheckExact(o)) return 0;
    const double d = PyLong_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return 0;
    *v = (float)d;
    return 1;
}

/* gemm_ex(address of vkblas_gemm_ex_async, its 23 arguments up to split_k,
 * use_epilogue, c_in, ldc_in, stride_c_in, bias, bias_type, stream) */
enum { NARGS = 31 };
static PyObject* gemm_ex(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    (void)self;
    if (n != NARGS) return PyErr_Format(PyExc_TypeError, "gemm_ex takes %d arguments (%zd given)", (int)NARGS, n);
    /* i: int, p: pointer, f: float, in the order of the arguments */
    static const char kind[] = "piiiiiiifpipifpiiiiiippiipiipip";
    unsigned long long v[NARGS];
    float alpha = 0.0f, beta = 0.0f;
    for (int k = 0; k < NARGS; ++k) {
        const int ok = kind[k] == 'i' ? get_int(a[k], &v[k])
                     : kind[k] == 'p' ? get_ptr(a[k], &v[k]) : get_float(a[k], k == 8 ? &alpha : &beta);
        if (!ok) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
    }
    if (!v[0]) return PyErr_Format(PyExc_ValueError, "no function address");
    const gemm_ex_fn fn = (gemm_ex_fn)(uintptr_t)v[0];
    vkblas_epilogue_t ep = {(const void*)(uintptr_t)v[25], (uint32_t)v[26], (int64_t)v[27],
                            (const void*)(uintptr_t)v[28], (vkblas_dtype_t)(int)v[29]};
    int st;
    Py_BEGIN_ALLOW_THREADS
    st = (int)fn((vkblas_dtype_t)(int)v[1], (vkblas_dtype_t)(int)v[2], (vkblas_op_t)(int)v[3], (vkblas_op_t)(int)v[4],
                 (uint32_t)v[5], (uint32_t)v[6], (uint32_t)v[7], alpha, (const void*)(uintptr_t)v[9], (uint32_t)v[10],
                 (const void*)(uintptr_t)v[11], (uint32_t)v[12], beta, (void*)(uintptr_t)v[14], (uint32_t)v[15],
                 (uint32_t)v[16], (int64_t)v[17], (int64_t)v[18], (int64_t)v[19], (vkblas_scalar_mode_t)(int)v[20],
                 (const void*)(uintptr_t)v[21], (const void*)(uintptr_t)v[22], (uint32_t)v[23], v[24] ? &ep : NULL,
                 (void*)(uintptr_t)v[30]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(st);
}

static PyMethodDef methods[] = {{"gemm_ex", (PyCFunction)(void (*)(void))gemm_ex, METH_FASTCALL,
                                 "vkblas_gemm_ex_async by address; None if an argument is not a plain int, float or None"},
                                {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", "GEMM calls of the binding", -1, methods,
                                    NULL, NULL, NULL, NULL};
PyMODINIT_FUNC PyInit__call(void) { return PyModule_Create(&module); }
