// The Python front-ends gemm, gemm_strided_batched and gemm_strided_batched_static_workspace as functions of a CPython module: a call goes from the
// interpreter's argument array to the C ABI without ctypes objects in between.  What a small GEMM costs a Python program is the host: of 5.1 us
// for 64 x 64 x 64 (api.py's own functions) 2.4 are the launch, and 1.7 went into arguments (a call that returns for m = 0).
//
// Only plain calls are taken here -- positional arguments, int, float, None, and objects with data_ptr() or cuda_stream.  Everything else,
// and any conversion that fails, goes to the Python function of the same name with the arguments as they came: one place decides
// what is accepted and which error is raised.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stddef.h>
#include <stdint.h>

namespace {

typedef int (*gemm_fn)(int, int, int, size_t, size_t, size_t, const void *, const void *, size_t, const void *, size_t, const void *, void *, size_t, int, void *);
typedef int (*batched_fn)(int, int, int, size_t, size_t, size_t, const void *, const void *, size_t, long long, const void *, size_t, long long, const void *,
                          void *, size_t, long long, int, int, void *);

constexpr long kF64 = 2;

gemm_fn g_gemm = nullptr;                       // set by bind(), once the library is loaded; read and written under the GIL
batched_fn g_batched = nullptr, g_static = nullptr;
PyObject *g_python[3] = {};                     // the Python functions
PyObject *g_check = nullptr;                    // raises what a status stands for
PyObject *g_data_ptr = nullptr, *g_cuda_stream = nullptr;   // names

// (masked to the width of the C argument, as ctypes does: a negative size is a huge one, which the library refuses)
inline bool integer(PyObject *o, unsigned long long *v)
{
    if (!PyLong_Check(o)) return false;
    *v = PyLong_AsUnsignedLongLongMask(o);
    return true;
}
inline bool address(PyObject *o, PyObject *name, bool call, void **p)
{
    if (o == Py_None) { *p = nullptr; return true; }
    unsigned long long v;
    if (integer(o, &v)) { *p = (void *)(uintptr_t)v; return true; }
    PyObject *r = call ? PyObject_CallMethodNoArgs(o, name) : PyObject_GetAttr(o, name);
    if (!r) { PyErr_Clear(); return false; }
    const bool ok = integer(r, &v);
    Py_DECREF(r);
    *p = (void *)(uintptr_t)v;
    return ok;
}
struct Scalar {
    union { float f; double d; };
};
inline bool scalar(PyObject *o, bool f64, Scalar *s)
{
    double v;
    if (PyFloat_CheckExact(o)) v = PyFloat_AS_DOUBLE(o);
    else if (PyLong_CheckExact(o)) {
        v = PyLong_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    } else return false;
    if (f64) s->d = v;
    else s->f = (float)v;
    return true;
}

// which: 0 gemm, 1 gemm_strided_batched, 2 its form with the static workspace.  1: not a plain call.
int plain_call(int which, PyObject *const *a, Py_ssize_t n, int *status)
{
    const Py_ssize_t need = which == 0 ? 14 : 18;
    if (n < need || n > need + 2 || (which == 0 ? !g_gemm : which == 1 ? !g_batched : !g_static)) return 1;
    unsigned long long i[6], lda, ldb, ldc, sa = 0, sb = 0, sc = 0, batch = 1, config = (unsigned long long)-1;
    for (int q = 0; q < 6; ++q)
        if (!integer(a[q], &i[q])) return 1;
    // (ctypes front-ends compare the Python value with F64)
    const bool f64 = (long long)i[0] == kF64;
    if (f64 != ((int)i[0] == (int)kF64)) return 1;
    Scalar alpha, beta;
    void *A, *B, *C, *stream = nullptr;
    Py_ssize_t at = 6;
    if (!scalar(a[at++], f64, &alpha) || !address(a[at++], g_data_ptr, true, &A) || !integer(a[at++], &lda)) return 1;
    if (which != 0 && !integer(a[at++], &sa)) return 1;
    if (!address(a[at++], g_data_ptr, true, &B) || !integer(a[at++], &ldb)) return 1;
    if (which != 0 && !integer(a[at++], &sb)) return 1;
    if (!scalar(a[at++], f64, &beta) || !address(a[at++], g_data_ptr, true, &C) || !integer(a[at++], &ldc)) return 1;
    if (which != 0 && (!integer(a[at++], &sc) || !integer(a[at++], &batch))) return 1;
    if (at < n && !integer(a[at++], &config)) return 1;
    if (at < n && !address(a[at++], g_cuda_stream, false, &stream)) return 1;
    const gemm_fn gemm = g_gemm;
    const batched_fn batched = which == 1 ? g_batched : g_static;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = which == 0 ? gemm((int)i[0], (int)i[1], (int)i[2], i[3], i[4], i[5], &alpha, A, lda, B, ldb, &beta, C, ldc, (int)config, stream)
                    : batched((int)i[0], (int)i[1], (int)i[2], i[3], i[4], i[5], &alpha, A, lda, (long long)sa, B, ldb, (long long)sb, &beta, C, ldc,
                              (long long)sc, (int)batch, (int)config, stream);
    Py_END_ALLOW_THREADS
    *status = rc;
    return 0;
}

template <int WHICH>
PyObject *front_end(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames)
{
    int status = 0;
    if (kwnames == nullptr && plain_call(WHICH, args, nargs, &status) == 0) {
        if (status == 0) Py_RETURN_NONE;
        return PyObject_CallFunction(g_check, "i", status);
    }
    if (!g_python[WHICH]) {
        PyErr_SetString(PyExc_RuntimeError, "not set up");
        return nullptr;
    }
    return PyObject_Vectorcall(g_python[WHICH], args, (size_t)nargs, kwnames);
}

// setup(gemm, gemm_strided_batched, gemm_strided_batched_static_workspace, check): the Python functions
PyObject *setup(PyObject *, PyObject *args)
{
    PyObject *f[3], *check;
    if (!PyArg_ParseTuple(args, "OOOO", &f[0], &f[1], &f[2], &check)) return nullptr;
    for (int q = 0; q < 3; ++q) {
        Py_INCREF(f[q]);
        Py_XSETREF(g_python[q], f[q]);
    }
    Py_INCREF(check);
    Py_XSETREF(g_check, check);
    Py_RETURN_NONE;
}

// bind(gemm, batched, static): addresses of the library's functions
PyObject *bind(PyObject *, PyObject *args)
{
    unsigned long long a, b, c;
    if (!PyArg_ParseTuple(args, "KKK", &a, &b, &c)) return nullptr;
    g_gemm = (gemm_fn)(uintptr_t)a;
    g_batched = (batched_fn)(uintptr_t)b;
    g_static = (batched_fn)(uintptr_t)c;
    Py_RETURN_NONE;
}

#define FRONT_END(name, which, rest) \
    {name, (PyCFunction)(void (*)(void))front_end<which>, METH_FASTCALL | METH_KEYWORDS, name rest}
PyMethodDef methods[] = {
    FRONT_END("gemm", 0, "(dtype, transA, transB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, config_id=-1, stream=None)\n--\n\n"
              "C = alpha*op(A)*op(B) + beta*C on the current device; asynchronous on `stream`."),
    FRONT_END("gemm_strided_batched", 1, "(dtype, transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC, batch, "
              "config_id=-1, stream=None)\n--\n\n"),
    FRONT_END("gemm_strided_batched_static_workspace", 2, "(dtype, transA, transB, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, "
              "strideC, batch, config_id=-1, stream=None)\n--\n\n"
              "The same GEMM without any device allocation: split-K partial sums go to the library's static per-device array\n"
              "(static_workspace_bytes() of them); a call that needs more raises MmboError with status 8."),
    {"setup", setup, METH_VARARGS, nullptr},
    {"bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_frontend", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__frontend(void)
{
    g_data_ptr = PyUnicode_InternFromString("data_ptr");
    g_cuda_stream = PyUnicode_InternFromString("cuda_stream");
    if (!g_data_ptr || !g_cuda_stream) return nullptr;
    return PyModule_Create(&module);
}
