// The calls of a program's inner loop - Plan.gemm and Plan.lstm_step - from Python to libtwgemm without ctypes, which takes 0.1 us
// and more to turn each of a dozen arguments, and the wrappers in Python as long again: a call on a few rows of A is
// little else.  From Python up to the library (a call that has nothing to do): `Plan.gemm` 2.2 us, with bias and
// workspace 3.2, `lstm_step` 3.0; this way 0.38, 0.44 and 0.45.  VGG16 conv4_1 for five images, a call after the other: 8.1 -> 7.5 us.
// The functions' addresses come from the library that twgemm.py has loaded; arguments that are no plain
// int, float, truth value or None are left to ctypes, which takes or refuses them as ever (None is returned then).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>

#include "twgemm.h"

namespace {

decltype(&tw_gemm_ex) g_gemm_ex = nullptr;
decltype(&tw_gemm_static) g_gemm_static = nullptr;
decltype(&tw_gemm_staged) g_gemm_staged = nullptr;
decltype(&tw_lstm_step) g_lstm_step = nullptr;

// Arguments one after the other; `ok` goes to false at the first that is not a plain one.
struct Args {
    PyObject *const *at;
    bool ok = true;
    explicit Args(PyObject *const *args) : at(args) {}
    uint64_t bits()
    {
        PyObject *o = *at++;
        if (!PyLong_CheckExact(o)) {
            ok = false;
            return 0;
        }
        return PyLong_AsUnsignedLongLongMask(o); // (as ctypes: the low bits of whatever is given)
    }
    int i32() { return (int)(uint32_t)bits(); }
    int64_t i64() { return (int64_t)bits(); }
    // an address, or None
    void *address()
    {
        if (*at == Py_None) {
            ++at;
            return nullptr;
        }
        return reinterpret_cast<void *>((uintptr_t)bits());
    }
    float f32()
    {
        PyObject *o = *at++;
        if (PyFloat_CheckExact(o))
            return (float)PyFloat_AS_DOUBLE(o);
        double v = 0.0;
        if (!PyLong_CheckExact(o) || ((v = PyLong_AsDouble(o)) == -1.0 && PyErr_Occurred())) {
            PyErr_Clear();
            ok = false;
        }
        return (float)v;
    }
};

bool number_of(PyObject *o, uintptr_t *out)
{
    const unsigned long long v = PyLong_AsUnsignedLongLong(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred())
        return false;
    *out = (uintptr_t)v;
    return true;
}

// bind(tw_gemm_ex, tw_gemm_static, tw_gemm_staged, tw_lstm_step): their addresses
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    uintptr_t a[4];
    if (n != 4) {
        PyErr_SetString(PyExc_TypeError, "four addresses");
        return nullptr;
    }
    for (int i = 0; i < 4; ++i)
        if (!number_of(args[i], &a[i]))
            return nullptr;
    g_gemm_ex = reinterpret_cast<decltype(g_gemm_ex)>(a[0]);
    g_gemm_static = reinterpret_cast<decltype(g_gemm_static)>(a[1]);
    g_gemm_staged = reinterpret_cast<decltype(g_gemm_staged)>(a[2]);
    g_lstm_step = reinterpret_cast<decltype(g_lstm_step)>(a[3]);
    Py_RETURN_NONE;
}

// gemm(plan, A, a_layout, lda, C, c_layout, ldc, M, alpha, beta, pruned_cols, stream, bias, activation, static, workspace,
// workspace_bytes): the status
PyObject *gemm(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 17 || !g_gemm_ex)
        Py_RETURN_NONE;
    Args in(args);
    const tw_plan *plan = static_cast<const tw_plan *>(in.address());
    const void *A = in.address();
    const int a_layout = in.i32();
    const int64_t lda = in.i64();
    void *C = in.address();
    const int c_layout = in.i32();
    const int64_t ldc = in.i64();
    const int M = in.i32();
    const float alpha = in.f32(), beta = in.f32();
    const int pruned = in.i32();
    void *stream = in.address();
    tw_epilogue ep;
    ep.bias = static_cast<const float *>(in.address());
    ep.activation = in.i32();
    PyObject *const fixed = *in.at++;
    const bool staged = *in.at != Py_None;
    void *workspace = in.address();
    const int64_t workspace_bytes = in.i64();
    if (!in.ok || (fixed != Py_True && fixed != Py_False))
        Py_RETURN_NONE;
    int status;
    Py_BEGIN_ALLOW_THREADS;
    if (staged)
        status = g_gemm_staged(plan, A, a_layout, lda, C, c_layout, ldc, M, alpha, beta, pruned, &ep, workspace, workspace_bytes, stream);
    else
        status = (fixed == Py_True ? g_gemm_static : g_gemm_ex)(plan, A, a_layout, lda, C, c_layout, ldc, M, alpha, beta, pruned, &ep, stream);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(status);
}

// lstm_step(plan, A, lda, M, bias, forget_bias, c_prev, ldc_prev, c_new, ldc_new, h_new, ldh, gates, ldg, stream): the status
PyObject *lstm_step(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 15 || !g_lstm_step)
        Py_RETURN_NONE;
    Args in(args);
    const tw_plan *plan = static_cast<const tw_plan *>(in.address());
    const void *A = in.address();
    const int64_t lda = in.i64();
    const int M = in.i32();
    const float *bias = static_cast<const float *>(in.address());
    const float forget_bias = in.f32();
    const float *c_prev = static_cast<const float *>(in.address());
    const int64_t ldc_prev = in.i64();
    float *c_new = static_cast<float *>(in.address());
    const int64_t ldc_new = in.i64();
    void *h_new = in.address();
    const int64_t ldh = in.i64();
    void *gates = in.address();
    const int64_t ldg = in.i64();
    void *stream = in.address();
    if (!in.ok)
        Py_RETURN_NONE;
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = g_lstm_step(plan, A, lda, M, bias, forget_bias, c_prev, ldc_prev, c_new, ldc_new, h_new, ldh, gates, ldg, stream);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(status);
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL, nullptr},
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gemm)), METH_FASTCALL, nullptr},
    {"lstm_step", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(lstm_step)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_twcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__twcall() { return PyModule_Create(&module); }
