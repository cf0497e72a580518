/* The calls of capi.py that a program makes in its inner loop - one multiply, one update of a plan's values - from Python
 * objects to the C-ABI in one step: addresses and sizes are taken from the tensors and the stream is looked up here.
 * Through ctypes, with one Python expression per argument, a multiply of a matrix that takes 2.5 us on the device took
 * 9.4 us; so it takes about half of that.  The library's functions are passed as addresses: this module links
 * against nothing. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stddef.h>
#include <stdint.h>

typedef int (*spmv64_t)(const void *, int, int32_t, int32_t, int32_t, double, const int32_t *, const int32_t *, const double *,
                        const double *, double, double *, void *, size_t, void *);
typedef int (*spmv32_t)(const void *, int, int32_t, int32_t, int32_t, float, const int32_t *, const int32_t *, const float *,
                        const float *, float, float *, void *, size_t, void *);
typedef int (*spmm64_t)(const void *, int, int32_t, int32_t, int32_t, int32_t, double, const int32_t *, const int32_t *,
                        const double *, const double *, int64_t, double, double *, int64_t, void *, size_t, void *);
typedef int (*spmm32_t)(const void *, int, int32_t, int32_t, int32_t, int32_t, float, const int32_t *, const int32_t *,
                        const float *, const float *, int64_t, float, float *, int64_t, void *, size_t, void *);
typedef int (*values_t)(void *, const void *, void *);

static PyObject *s_data_ptr, *s_numel, *s_element_size;
static PyObject *get_device, *get_stream; /* the current device's number; the stream of a device, as an integer */

/* result of a method without arguments, as an integer; -1 with an exception set on failure */
static int64_t ask(PyObject *o, PyObject *method)
{
    PyObject *r = PyObject_CallMethodNoArgs(o, method);
    if (!r) return -1;
    const int64_t v = (int64_t)PyLong_AsUnsignedLongLongMask(r);
    Py_DECREF(r);
    return v;
}
static void *address(PyObject *o) { return o == Py_None ? NULL : (void *)(uintptr_t)ask(o, s_data_ptr); }
static int64_t number(PyObject *o) { return PyLong_AsLongLong(o); }
static void *pointer(PyObject *o) { return o == Py_None ? NULL : (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(o); }

static void *stream(void)
{
    PyObject *d = PyObject_CallNoArgs(get_device);
    if (!d) return NULL;
    PyObject *r = PyObject_CallOneArg(get_stream, d);
    Py_DECREF(d);
    if (!r) return NULL;
    void *s = (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(r);
    Py_DECREF(r);
    return s;
}

static PyObject *streams_from(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    (void)self;
    if (n != 2) return PyErr_Format(PyExc_TypeError, "streams_from(get_device, get_stream)");
    Py_INCREF(a[0]);
    Py_INCREF(a[1]);
    Py_XSETREF(get_device, a[0]);
    Py_XSETREF(get_stream, a[1]);
    Py_RETURN_NONE;
}

/* int32 argument: sizes beyond it are an error, as they are for ctypes' c_int32 callers that check */
static int32_t size32(int64_t v)
{
    if ((v < INT32_MIN || v > INT32_MAX) && !PyErr_Occurred()) PyErr_Format(PyExc_OverflowError, "%lld does not fit int32", (long long)v);
    return (int32_t)v;
}

/* workspace: None (no buffer) or a tensor */
static void workspace_of(PyObject *o, void **p, size_t *bytes)
{
    *p = NULL;
    *bytes = 0;
    if (o == Py_None) return;
    *p = address(o);
    *bytes = (size_t)(ask(o, s_numel) * ask(o, s_element_size));
}

/* spmv(fn, f64, plan, alg, row_ptr, col, val, x, y, alpha, beta, n or None, workspace or None) -> status */
static PyObject *spmv(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    (void)self;
    if (n != 13 || !get_stream) return PyErr_Format(PyExc_TypeError, "spmv: 13 arguments, after streams_from");
    void *fn = pointer(a[0]), *plan = pointer(a[2]), *ws;
    const int f64 = a[1] == Py_True, alg = (int)number(a[3]);
    size_t ws_bytes;
    const int32_t m = size32(ask(a[4], s_numel) - 1), nnz = size32(ask(a[5], s_numel));
    const int32_t cols = size32(a[11] == Py_None ? ask(a[7], s_numel) : number(a[11]));
    const int32_t *rp = address(a[4]), *col = address(a[5]);
    const void *val = address(a[6]), *x = address(a[7]);
    void *y = address(a[8]);
    const double alpha = PyFloat_AsDouble(a[9]), beta = PyFloat_AsDouble(a[10]);
    workspace_of(a[12], &ws, &ws_bytes);
    void *s = stream();
    if (PyErr_Occurred()) return NULL;
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = f64 ? ((spmv64_t)fn)(plan, alg, m, cols, nnz, alpha, rp, col, val, x, beta, y, ws, ws_bytes, s)
             : ((spmv32_t)fn)(plan, alg, m, cols, nnz, (float)alpha, rp, col, val, x, (float)beta, y, ws, ws_bytes, s);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(st);
}

/* spmm(fn, f64, plan, alg, row_ptr, col, val, B, C, ncols, alpha, beta, ldb or None, ldc or None, k or None, workspace or None) -> status */
static PyObject *spmm(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    (void)self;
    if (n != 16 || !get_stream) return PyErr_Format(PyExc_TypeError, "spmm: 16 arguments, after streams_from");
    void *fn = pointer(a[0]), *plan = pointer(a[2]), *ws;
    const int f64 = a[1] == Py_True, alg = (int)number(a[3]);
    size_t ws_bytes;
    const int32_t m = size32(ask(a[4], s_numel) - 1), nnz = size32(ask(a[5], s_numel)), ncols = size32(number(a[9]));
    const int64_t ldb = a[12] == Py_None ? ncols : number(a[12]), ldc = a[13] == Py_None ? ncols : number(a[13]);
    int64_t rows = 0;
    if (a[14] != Py_None)
        rows = number(a[14]);
    else if (ldb != 0)
        rows = ask(a[7], s_numel) / ldb;
    else
        PyErr_SetString(PyExc_ZeroDivisionError, "spmm: ldb = 0");
    const int32_t k = size32(rows);
    const int32_t *rp = address(a[4]), *col = address(a[5]);
    const void *val = address(a[6]), *B = address(a[7]);
    void *C = address(a[8]);
    const double alpha = PyFloat_AsDouble(a[10]), beta = PyFloat_AsDouble(a[11]);
    workspace_of(a[15], &ws, &ws_bytes);
    void *s = stream();
    if (PyErr_Occurred()) return NULL;
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = f64 ? ((spmm64_t)fn)(plan, alg, m, k, nnz, ncols, alpha, rp, col, val, B, ldb, beta, C, ldc, ws, ws_bytes, s)
             : ((spmm32_t)fn)(plan, alg, m, k, nnz, ncols, (float)alpha, rp, col, val, B, ldb, (float)beta, C, ldc, ws, ws_bytes, s);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(st);
}

/* plan_values(fn, plan, val) -> status of fn(plan, val, stream) */
static PyObject *plan_values(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    (void)self;
    if (n != 3 || !get_stream) return PyErr_Format(PyExc_TypeError, "plan_values: 3 arguments, after streams_from");
    void *fn = pointer(a[0]), *plan = pointer(a[1]), *val = address(a[2]), *s = stream();
    if (PyErr_Occurred()) return NULL;
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = ((values_t)fn)(plan, val, s);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(st);
}

static PyMethodDef methods[] = {
    {"streams_from", (PyCFunction)(void (*)(void))streams_from, METH_FASTCALL, "callables for the current device and a device's stream"},
    {"spmv", (PyCFunction)(void (*)(void))spmv, METH_FASTCALL, "asx_spmv_csr_*"},
    {"spmm", (PyCFunction)(void (*)(void))spmm, METH_FASTCALL, "asx_spmm_csr_*"},
    {"plan_values", (PyCFunction)(void (*)(void))plan_values, METH_FASTCALL, "asx_plan_update_values, asx_plan_refresh_if_changed"},
    {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "calls into libalphasparse_amd.so", -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__calls(void)
{
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_numel = PyUnicode_InternFromString("numel");
    s_element_size = PyUnicode_InternFromString("element_size");
    if (!s_data_ptr || !s_numel || !s_element_size) return NULL;
    return PyModule_Create(&module);
}
