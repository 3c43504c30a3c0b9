// The calls of a serving loop, from Python: the GEMM and the quantisers take a few microseconds on the device, and a
// ctypes call with nine arguments and five look-ups of a pointer take 1.4 us on the host, which is what a small call waits
// for (calls back to back, through ctypes / from here: a GEMM 4.9 / 4.3 us, quantiser and GEMM 9.4 / 7.7 us).  These functions take what such a loop passes -- tensors (anything with data_ptr()), plain
// integers and None -- and answer None to everything else: the caller then goes through ctypes, whose conversions and
// errors stay the only ones.  The lock of the interpreter is given up during the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/fp8_block_gemm.h"

namespace {

PyObject* g_data_ptr;      // the name "data_ptr"
PyObject* g_options_type;  // the Options structure, set once by setup()

// a device pointer as ctypes takes it: None, an int (its low 64 bits), or data_ptr() of anything else
bool pointer(PyObject* x, void** out)
{
    if (x == Py_None) {
        *out = nullptr;
        return true;
    }
    if (PyLong_CheckExact(x)) {
        *out = reinterpret_cast<void*>(PyLong_AsUnsignedLongLongMask(x));
        return true;
    }
    if (PyLong_Check(x))
        return false;
    PyObject* p = PyObject_CallMethodNoArgs(x, g_data_ptr);
    if (!p) {
        PyErr_Clear();
        return false;
    }
    const bool ok = PyLong_CheckExact(p);
    if (ok)
        *out = reinterpret_cast<void*>(PyLong_AsUnsignedLongLongMask(p));
    Py_DECREF(p);
    return ok;
}

bool pointers(PyObject* const* args, int count, void** out)
{
    for (int i = 0; i < count; ++i)
        if (!pointer(args[i], &out[i]))
            return false;
    return true;
}

bool integers(PyObject* const* args, int count, int* out)
{
    for (int i = 0; i < count; ++i) {
        if (!PyLong_CheckExact(args[i]))
            return false;
        out[i] = (int)PyLong_AsUnsignedLongMask(args[i]);
    }
    return true;
}

// a stream: an int or None, no tensor
bool stream(PyObject* x, void** out) { return (x == Py_None || PyLong_CheckExact(x)) && pointer(x, out); }

// gemm(a, b, a_scale, b_scale, c, m, n, k, stream)
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    void *p[5], *s;
    int d[3], rc;
    if (count != 9 || !pointers(args, 5, p) || !integers(args + 5, 3, d) || !stream(args[8], &s))
        Py_RETURN_NONE;
    Py_BEGIN_ALLOW_THREADS
    rc = fp8_block_gemm_stream(p[0], p[1], static_cast<float*>(p[2]), static_cast<float*>(p[3]), p[4], d[0], d[1], d[2], s);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

// gemm_ex(a, b, a_scale, b_scale, c, m, n, k, options, workspace, workspace_bytes, stream)
PyObject* gemm_ex(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    void *p[5], *s, *ws;
    int d[3], rc;
    if (count != 12 || !pointers(args, 5, p) || !integers(args + 5, 3, d) || !pointer(args[9], &ws) ||
        !PyLong_CheckExact(args[10]) || !stream(args[11], &s))
        Py_RETURN_NONE;
    const size_t bytes = (size_t)PyLong_AsUnsignedLongMask(args[10]);
    Py_buffer view;
    view.obj = nullptr;
    const fp8gemm_options* options = nullptr;
    if (args[8] != Py_None) {
        if ((PyObject*)Py_TYPE(args[8]) != g_options_type)
            Py_RETURN_NONE;
        if (PyObject_GetBuffer(args[8], &view, PyBUF_SIMPLE) != 0) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        if (view.len != (Py_ssize_t)sizeof(fp8gemm_options)) {
            PyBuffer_Release(&view);
            Py_RETURN_NONE;
        }
        options = static_cast<const fp8gemm_options*>(view.buf);
    }
    Py_BEGIN_ALLOW_THREADS
    rc = fp8_block_gemm_ex(p[0], p[1], static_cast<float*>(p[2]), static_cast<float*>(p[3]), p[4], d[0], d[1], d[2], options, ws, bytes, s);
    Py_END_ALLOW_THREADS
    if (view.obj)
        PyBuffer_Release(&view);
    return PyLong_FromLong(rc);
}

// quantize_a(x, dtype, q, scale, rows, k, stream), quantize_b likewise
template <int (*CALL)(const void*, int, void*, float*, int, int, void*)>
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    void *x, *q, *scale, *s;
    int dtype, d[2], rc;
    if (count != 7 || !pointer(args[0], &x) || !integers(args + 1, 1, &dtype) || !pointer(args[2], &q) || !pointer(args[3], &scale) ||
        !integers(args + 4, 2, d) || !stream(args[6], &s))
        Py_RETURN_NONE;
    Py_BEGIN_ALLOW_THREADS
    rc = CALL(x, dtype, q, static_cast<float*>(scale), d[0], d[1], s);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

PyObject* setup(PyObject*, PyObject* options_type)
{
    Py_INCREF(options_type);
    Py_XDECREF(g_options_type);
    g_options_type = options_type;
    Py_RETURN_NONE;
}

template <class F>
constexpr PyCFunction fast(F f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

PyMethodDef methods[] = {
    {"setup", setup, METH_O, "setup(Options): the structure that gemm_ex takes"},
    {"gemm", fast(gemm), METH_FASTCALL, "the return code of fp8_block_gemm_stream, or None: not for this path"},
    {"gemm_ex", fast(gemm_ex), METH_FASTCALL, "the return code of fp8_block_gemm_ex, or None: not for this path"},
    {"quantize_a", fast(quantize<fp8_quantize_a_1x128>), METH_FASTCALL, "the return code of fp8_quantize_a_1x128, or None"},
    {"quantize_b", fast(quantize<fp8_quantize_b_128x128>), METH_FASTCALL, "the return code of fp8_quantize_b_128x128, or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pycall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pycall(void)
{
    g_data_ptr = PyUnicode_InternFromString("data_ptr");
    return g_data_ptr ? PyModule_Create(&module) : nullptr;
}
