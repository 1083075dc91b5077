/* py_call.c -- the package's launching calls without ctypes: one C function per entry point of
 * include/mi_gemm.h that launches.  ctypes converts eight to fourteen arguments through from_param
 * objects and the wrapper asks every operand what kind it is: 1.9 us of a 512^3 call's 4.3, whose
 * kernel takes 3.2.  Only the usual arguments are taken (Python ints within 32 bits, floats,
 * pointers as None, int, the package's DeviceBuffer or anything with data_ptr(), streams as None or
 * int); for any other the function returns None having done nothing, and the caller takes the
 * ctypes path with its conversions and errors. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <limits.h>
#include <stdint.h>

#include "../../include/mi_gemm.h"

static PyObject *s_data_ptr, *s_ptr, *device_buffer;

/* 1: converted, 0: not one of the usual kinds (no exception left set) */
static int to_int(PyObject* o, int* out) {
    int overflow = 0;
    if (!PyLong_CheckExact(o)) return 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    if (overflow || v < INT_MIN || v > INT_MAX) return 0;
    *out = (int)v;
    return 1;
}
static int to_float(PyObject* o, float* out) {
    if (!PyFloat_CheckExact(o)) return 0;
    *out = (float)PyFloat_AS_DOUBLE(o);
    return 1;
}
static int to_address(PyObject* o, void** out) {
    const unsigned long long v = PyLong_AsUnsignedLongLong(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) {
        PyErr_Clear();
        return 0;
    }
    *out = (void*)(uintptr_t)v;
    return 1;
}
/* (a pointer of 0 is NULL, as through ctypes) */
static int to_pointer(PyObject* o, void** out) {
    if (o == Py_None) {
        *out = NULL;
        return 1;
    }
    if (PyLong_CheckExact(o)) return to_address(o, out);
    PyObject* v = (PyObject*)Py_TYPE(o) == device_buffer ? PyObject_GetAttr(o, s_ptr) : PyObject_CallMethodNoArgs(o, s_data_ptr);
    if (v == NULL) {
        PyErr_Clear();
        return 0;
    }
    const int ok = PyLong_CheckExact(v) && to_address(v, out);
    Py_DECREF(v);
    return ok;
}
static int to_stream(PyObject* o, void** out) { return (o == Py_None || PyLong_CheckExact(o)) && to_pointer(o, out); }

#define NOT_USUAL Py_RETURN_NONE
#define INTS(n) for (int i = 0; i < (n); ++i) if (!to_int(a[i], &v[i])) NOT_USUAL
#define PTRS(from, n) for (int i = 0; i < (n); ++i) if (!to_pointer(a[(from) + i], &p[i])) NOT_USUAL
#define CALL(expr)                       \
    Py_BEGIN_ALLOW_THREADS rc = (expr);  \
    Py_END_ALLOW_THREADS return PyLong_FromLong(rc)

/* (M, N, K, A, B, C, DB, stream) */
static PyObject* call_bf16(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    int v[3], rc;
    void *p[4], *s;
    (void)self;
    if (n != 8) NOT_USUAL;
    INTS(3);
    PTRS(3, 4);
    if (!to_stream(a[7], &s)) NOT_USUAL;
    CALL(mi_gemm_bf16(v[0], v[1], v[2], (const uint16_t*)p[0], (const uint16_t*)p[1], (uint16_t*)p[2], (int*)p[3], s));
}
/* (config, dtype, M, N, K, A, B, C, DB, stream) */
static PyObject* call_ex(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    int v[5], rc;
    void *p[4], *s;
    (void)self;
    if (n != 10) NOT_USUAL;
    INTS(5);
    PTRS(5, 4);
    if (!to_stream(a[9], &s)) NOT_USUAL;
    CALL(mi_gemm_ex(v[0], v[1], v[2], v[3], v[4], p[0], p[1], p[2], (int*)p[3], s));
}
/* (config, dtype, M, N, K, A, B, C, alpha, beta, c_layout, stream) */
static PyObject* call_epilogue(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    int v[5], layout, rc;
    float alpha, beta;
    void *p[3], *s;
    (void)self;
    if (n != 12) NOT_USUAL;
    INTS(5);
    PTRS(5, 3);
    if (!to_float(a[8], &alpha) || !to_float(a[9], &beta) || !to_int(a[10], &layout) || !to_stream(a[11], &s)) NOT_USUAL;
    CALL(mi_gemm_epilogue(v[0], v[1], v[2], v[3], v[4], p[0], p[1], p[2], alpha, beta, layout, s));
}
/* (config, dtype, M, N, K, A, B, C, alpha, beta, c_layout, ws, ws_bytes, stream) */
static PyObject* call_epilogue_ws(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    int v[5], layout, rc;
    float alpha, beta;
    void *p[3], *ws, *bytes, *s;
    (void)self;
    if (n != 14) NOT_USUAL;
    INTS(5);
    PTRS(5, 3);
    if (!to_float(a[8], &alpha) || !to_float(a[9], &beta) || !to_int(a[10], &layout) || !to_stream(a[11], &ws) ||
        !PyLong_CheckExact(a[12]) || !to_address(a[12], &bytes) || !to_stream(a[13], &s))
        NOT_USUAL;
    CALL(mi_gemm_epilogue_ws(v[0], v[1], v[2], v[3], v[4], p[0], p[1], p[2], alpha, beta, layout, ws, (size_t)(uintptr_t)bytes, s));
}
/* (dtype, M, N, K, A, B, C, alpha, beta, stream) */
static PyObject* call_reference(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    int v[4], rc;
    float alpha, beta;
    void *p[3], *s;
    (void)self;
    if (n != 10) NOT_USUAL;
    INTS(4);
    PTRS(4, 3);
    if (!to_float(a[7], &alpha) || !to_float(a[8], &beta) || !to_stream(a[9], &s)) NOT_USUAL;
    CALL(mi_reference_gpu_gemm(v[0], v[1], v[2], v[3], p[0], p[1], p[2], alpha, beta, s));
}
/* the class whose `ptr` attribute is a device pointer */
static PyObject* set_device_buffer(PyObject* self, PyObject* cls) {
    (void)self;
    Py_INCREF(cls);
    Py_XSETREF(device_buffer, cls);
    Py_RETURN_NONE;
}

static PyMethodDef methods[] = {
    {"bf16", (PyCFunction)(void (*)(void))call_bf16, METH_FASTCALL, NULL},
    {"ex", (PyCFunction)(void (*)(void))call_ex, METH_FASTCALL, NULL},
    {"epilogue", (PyCFunction)(void (*)(void))call_epilogue, METH_FASTCALL, NULL},
    {"epilogue_ws", (PyCFunction)(void (*)(void))call_epilogue_ws, METH_FASTCALL, NULL},
    {"reference", (PyCFunction)(void (*)(void))call_reference, METH_FASTCALL, NULL},
    {"set_device_buffer", set_device_buffer, METH_O, NULL},
    {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "mi_py_call", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit_mi_py_call(void) {
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_ptr = PyUnicode_InternFromString("ptr");
    return s_data_ptr && s_ptr ? PyModule_Create(&module) : NULL;
}
