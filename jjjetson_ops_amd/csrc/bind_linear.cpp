// CPython binding of the two linear-layer entries for device tensors.
//
// A decode step's kernel takes 3 to 6 us, less than Python needs to pass four tensors
// through ctypes (7.1 us a call at K=4096, N=4096, whose kernel takes 3.5 us).  Here the
// tensors' attributes are read and the C entry is called in one native function.  No torch
// header is needed: is_cuda, is_contiguous() and data_ptr() are looked up on the object, the
// current stream comes from the callable that the Python side hands over once.
//
// linear(split, current_stream, x, w, y, in_features, out_features, num_tokens, ws, stream)
//   -> status code of linear_q4_0_forward_device / linear_q4_0s_forward_device, or None if a
//      size or an address is no int (the caller then leaves the conversion to ctypes)
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "jjjetson_ops_amd.h"

namespace {

PyObject *s_is_cuda, *s_is_contiguous, *s_data_ptr, *s_cuda_stream;

// An address as an int; -1 where it is none (no exception set).
int address(PyObject *r, void **out) {
    *out = PyLong_AsVoidPtr(r);
    if (*out != nullptr || !PyErr_Occurred()) return 1;
    PyErr_Clear();
    return -1;
}

// A C int as ctypes converts one (an int or an object with __index__, truncated); -1 for
// anything else: ctypes also takes its own c_int and _as_parameter_, and names the argument
// that it refuses.
int c_int(PyObject *o, int *out) {
    const unsigned long v = PyLong_AsUnsignedLongMask(o);
    *out = (int)v;
    if (v != (unsigned long)-1 || !PyErr_Occurred()) return 1;
    PyErr_Clear();
    return -1;
}

// The tensor's device address: 1, -1 (no int), or 0 with an exception set.
int device_ptr(PyObject *t, const char *name, void **out) {
    PyObject *r = PyObject_GetAttr(t, s_is_cuda);
    if (r == nullptr) return 0;
    int yes = PyObject_IsTrue(r);
    Py_DECREF(r);
    if (yes < 0) return 0;
    if (yes == 0) {
        PyErr_Format(PyExc_ValueError, "%s must be a device tensor", name);
        return 0;
    }
    if ((r = PyObject_CallMethodNoArgs(t, s_is_contiguous)) == nullptr) return 0;
    yes = PyObject_IsTrue(r);
    Py_DECREF(r);
    if (yes < 0) return 0;
    if (yes == 0) {
        PyErr_Format(PyExc_ValueError, "%s must be contiguous", name);
        return 0;
    }
    if ((r = PyObject_CallMethodNoArgs(t, s_data_ptr)) == nullptr) return 0;
    const int rc = address(r, out);
    Py_DECREF(r);
    return rc;
}

// None: the current stream; an int: a hipStream_t; anything else: its cuda_stream.
int stream_ptr(PyObject *stream, PyObject *current_stream, void **out) {
    PyObject *r;
    if (stream == Py_None)
        r = PyObject_CallNoArgs(current_stream);
    else if (PyLong_Check(stream))
        r = Py_NewRef(stream);
    else
        r = PyObject_GetAttr(stream, s_cuda_stream);
    if (r == nullptr) return 0;
    const int rc = address(r, out);
    Py_DECREF(r);
    return rc;
}

PyObject *linear(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 10) {
        PyErr_SetString(PyExc_TypeError, "linear takes 10 arguments");
        return nullptr;
    }
    const int split = PyObject_IsTrue(a[0]);
    if (split < 0) return nullptr;
    void *stream, *ws = nullptr, *x, *w, *y;
    int in, out, tokens;
    int rc = stream_ptr(a[9], a[1], &stream);
    if (rc > 0 && a[8] != Py_None) rc = device_ptr(a[8], "ws", &ws);
    if (rc > 0) rc = device_ptr(a[2], "x", &x);
    if (rc > 0) rc = device_ptr(a[3], "w", &w);
    if (rc > 0) rc = device_ptr(a[4], "y", &y);
    if (rc > 0) rc = c_int(a[5], &in);
    if (rc > 0) rc = c_int(a[6], &out);
    if (rc > 0) rc = c_int(a[7], &tokens);
    if (rc == 0) return nullptr;
    if (rc < 0) Py_RETURN_NONE;
    Py_BEGIN_ALLOW_THREADS
    rc = split ? linear_q4_0s_forward_device(stream, ws, (const float *)x, w, (float *)y, in, out, tokens)
               : linear_q4_0_forward_device(stream, ws, (const float *)x, w, (float *)y, in, out, tokens);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

PyMethodDef methods[] = {
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, "One linear layer on device tensors."},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_linear", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject *PyInit__linear(void) {
    s_is_cuda = PyUnicode_InternFromString("is_cuda");
    s_is_contiguous = PyUnicode_InternFromString("is_contiguous");
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_cuda_stream = PyUnicode_InternFromString("cuda_stream");
    if (s_is_cuda == nullptr || s_is_contiguous == nullptr || s_data_ptr == nullptr || s_cuda_stream == nullptr)
        return nullptr;
    return PyModule_Create(&module);
}
