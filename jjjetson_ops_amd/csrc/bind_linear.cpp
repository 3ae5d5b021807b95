// CPython binding of the two linear-layer entries for device tensors.
//
// A decode step's kernel takes 3 to 6 us, less than Python needs to pass four tensors
// through ctypes (7.1 us a call at K=4096, N=4096, whose kernel takes 3.5 us).  Here the
// tensors' attributes are read and the C entry is called in one native function.  No torch
// header is needed: is_cuda, is_contiguous() and data_ptr() are looked up on the object, the
// current stream comes from the callable that the Python side hands over once.
//
// linear(split, current_stream, x, w, y, in_features, out_features, num_tokens, ws, stream)
//   -> status code of linear_q4_0_forward_device / linear_q4_0s_forward_device
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "jjjetson_ops_amd.h"

namespace {

PyObject *s_is_cuda, *s_is_contiguous, *s_data_ptr, *s_cuda_stream;

// The tensor's device address; on failure returns false with an exception set.
bool device_ptr(PyObject *t, const char *name, void **out) {
    PyObject *r = PyObject_GetAttr(t, s_is_cuda);
    if (r == nullptr) return false;
    int yes = PyObject_IsTrue(r);
    Py_DECREF(r);
    if (yes < 0) return false;
    if (yes == 0) {
        PyErr_Format(PyExc_ValueError, "%s must be a device tensor", name);
        return false;
    }
    if ((r = PyObject_CallMethodNoArgs(t, s_is_contiguous)) == nullptr) return false;
    yes = PyObject_IsTrue(r);
    Py_DECREF(r);
    if (yes < 0) return false;
    if (yes == 0) {
        PyErr_Format(PyExc_ValueError, "%s must be contiguous", name);
        return false;
    }
    if ((r = PyObject_CallMethodNoArgs(t, s_data_ptr)) == nullptr) return false;
    *out = PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    return !(*out == nullptr && PyErr_Occurred());
}

// None: the current stream; an int: a hipStream_t; anything else: its cuda_stream.
bool stream_ptr(PyObject *stream, PyObject *current_stream, void **out) {
    PyObject *r;
    if (stream == Py_None)
        r = PyObject_CallNoArgs(current_stream);
    else if (PyLong_Check(stream))
        r = Py_NewRef(stream);
    else
        r = PyObject_GetAttr(stream, s_cuda_stream);
    if (r == nullptr) return false;
    *out = PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    return !(*out == nullptr && PyErr_Occurred());
}

// A C int as ctypes converts one (an int or an object with __index__, truncated).
bool c_int(PyObject *o, int *out) {
    const unsigned long v = PyLong_AsUnsignedLongMask(o);
    *out = (int)v;
    return !(v == (unsigned long)-1 && PyErr_Occurred());
}

PyObject *linear(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 10) {
        PyErr_SetString(PyExc_TypeError, "linear takes 10 arguments");
        return nullptr;
    }
    const int split = PyObject_IsTrue(a[0]);
    void *stream, *ws = nullptr, *x, *w, *y;
    int in, out, tokens;
    if (split < 0 || !stream_ptr(a[9], a[1], &stream) || (a[8] != Py_None && !device_ptr(a[8], "ws", &ws)) ||
        !device_ptr(a[2], "x", &x) || !device_ptr(a[3], "w", &w) || !device_ptr(a[4], "y", &y) || !c_int(a[5], &in) ||
        !c_int(a[6], &out) || !c_int(a[7], &tokens))
        return nullptr;
    int rc;
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
