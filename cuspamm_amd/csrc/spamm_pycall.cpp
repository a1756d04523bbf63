// The multiply calls of api.py for the usual arguments, without the interpreter's part of the checks.
//
// What a call costs on the host bounds the smallest ones: two launches are some 6.5 us, and the checks of three tensors, a parameter
// structure and a call through ctypes were 2.5 to 3 us more (256^3, whose kernels take 6.8 us, 9.6 us a call).  Here they are 0.4.
//
// Each function takes what api.py's method has been given and answers None -- unless everything is as it usually is: tensors and numbers
// of exactly the types expected, shapes that fit, one GPU, contiguous -- and api.py goes on by itself then, with its own checks
// and errors.  So it does where torch throws while a tensor is looked at (a size that is a symbol, say): nothing may be thrown through the
// interpreter's frames.  Otherwise the ABI's function has been called, with the interpreter released: the answer is its error code, or
// the shape tuple that the context keeps.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include "../../include/spamm.h"

namespace {

int (*g_multiply)(spamm_ctx *, const spamm_params *, const float *, const float *, float *);
int (*g_multiply_f16)(spamm_ctx *, const spamm_params *, const void *, const void *, float *);
int (*g_multiply_noalloc)(spamm_ctx *, const spamm_params *, const float *, const float *, float *);

const at::Tensor *matrix(PyObject *o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (t.is_nested() || t.dim() != 2 || !t.is_cuda() || t.layout() != c10::kStrided || !t.is_contiguous() || !t.has_storage() || t.is_neg() || t.is_conj()) return nullptr;
    return &t;
}

struct Call {
    spamm_ctx *ctx;
    spamm_params p;
    const void *a, *b;
    float *c;
    bool half;
};

// args: handle, A, B, C, tile, tau, flags (each a truth value: its bit).  False: not the usual arguments, or none that Python numbers
// or truth values can be had of (its error is set).
bool usual(PyObject *const *args, Py_ssize_t n, Py_ssize_t expected, const uint32_t *flag_bits, bool noalloc, Call &out) {
    if (n != expected || !g_multiply) return false;
    if (!PyLong_CheckExact(args[0]) || !PyLong_CheckExact(args[4]) || !(PyFloat_CheckExact(args[5]) || PyLong_CheckExact(args[5]))) return false;
    const at::Tensor *A = matrix(args[1]), *B = matrix(args[2]), *C = matrix(args[3]);
    if (!A || !B || !C) return false;
    const int64_t M = A->size(0), K = A->size(1), N = B->size(1);
    if (B->size(0) != K || C->size(0) != M || C->size(1) != N || A->device() != B->device() || A->device() != C->device()) return false;
    const at::ScalarType type = A->scalar_type();
    if (B->scalar_type() != type || C->scalar_type() != at::kFloat || (type != at::kFloat && (noalloc || type != at::kHalf))) return false;
    out.ctx = static_cast<spamm_ctx *>(PyLong_AsVoidPtr(args[0]));
    const long tile = PyLong_AsLong(args[4]);
    const double tau = PyFloat_AsDouble(args[5]);
    if (PyErr_Occurred() || !out.ctx || tile < 1 || tile > 128) return false;
    out.p = {};
    out.p.M = M;
    out.p.K = K;
    out.p.N = N;
    out.p.tile = (int32_t)tile;
    out.p.tau = (float)tau;
    for (Py_ssize_t i = 6; i < expected; i++) {
        const int on = PyObject_IsTrue(args[i]);
        if (on < 0) return false;
        if (on) out.p.flags |= flag_bits[i - 6];
    }
    out.a = A->const_data_ptr();
    out.b = B->const_data_ptr();
    out.c = static_cast<float *>(C->data_ptr());
    out.half = type == at::kHalf;
    return true;
}

PyObject *call(PyObject *const *args, Py_ssize_t n, Py_ssize_t expected, const uint32_t *flag_bits, bool noalloc) {
    Call k;
    bool go = false;
    try {
        go = usual(args, n, expected, flag_bits, noalloc, k);
    } catch (...) {
    }
    if (!go) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    int code;
    Py_BEGIN_ALLOW_THREADS
    if (noalloc) code = g_multiply_noalloc(k.ctx, &k.p, static_cast<const float *>(k.a), static_cast<const float *>(k.b), k.c);
    else if (k.half) code = g_multiply_f16(k.ctx, &k.p, k.a, k.b, k.c);
    else code = g_multiply(k.ctx, &k.p, static_cast<const float *>(k.a), static_cast<const float *>(k.b), k.c);
    Py_END_ALLOW_THREADS
    if (code != SPAMM_OK) return PyLong_FromLong(code);
    const long long M = k.p.M, K = k.p.K, N = k.p.N;
    const long tile = k.p.tile;
    return Py_BuildValue("(LLLlLLL)", M / tile, K / tile, N / tile, tile, M, K, N);
}

PyObject *multiply(PyObject *, PyObject *const *args, Py_ssize_t n) {
    static const uint32_t bits[] = {SPAMM_FLAG_TIMING, SPAMM_FLAG_REUSE_A, SPAMM_FLAG_REUSE_B, SPAMM_FLAG_A_EQ_B, SPAMM_FLAG_PRUNE};
    return call(args, n, 6 + 5, bits, false);
}

PyObject *multiply_noalloc(PyObject *, PyObject *const *args, Py_ssize_t n) {
    static const uint32_t bits[] = {SPAMM_FLAG_TIMING, SPAMM_FLAG_A_EQ_B, SPAMM_FLAG_PRUNE};
    return call(args, n, 6 + 3, bits, true);
}

// The loaded library's functions, by address
PyObject *bind(PyObject *, PyObject *args) {
    unsigned long long m, h, s;
    if (!PyArg_ParseTuple(args, "KKK", &m, &h, &s)) return nullptr;
    g_multiply = reinterpret_cast<decltype(g_multiply)>(m);
    g_multiply_f16 = reinterpret_cast<decltype(g_multiply_f16)>(h);
    g_multiply_noalloc = reinterpret_cast<decltype(g_multiply_noalloc)>(s);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"multiply", (PyCFunction)(void (*)(void))multiply, METH_FASTCALL, "handle, A, B, C, tile, tau, timing, reuse_a, reuse_b, a_eq_b, prune"},
    {"multiply_noalloc", (PyCFunction)(void (*)(void))multiply_noalloc, METH_FASTCALL, "handle, A, B, C, tile, tau, timing, a_eq_b, prune"},
    {"bind", bind, METH_VARARGS, "addresses of spamm_multiply, spamm_multiply_f16, spamm_multiply_noalloc"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_spamm_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: of the torch whose headers this was built with; with another one its tensors are not to be looked into
PyMODINIT_FUNC PyInit__spamm_call(void) {
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", SPAMM_TORCH_VERSION) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
