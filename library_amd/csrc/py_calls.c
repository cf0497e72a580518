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

static PyObject *s_data_ptr, *s_numel, *s_element_size, *s_dim, *s_size, *s_stride;
static PyObject *get_device, *get_stream; /* the current device's number; the stream of a device, as an integer */
static PyObject *argument_error;          /* ctypes.ArgumentError */

/* Each of these writes *out and returns 1, or leaves an exception set and returns 0, after which nothing else of Python may
 * be called: they are joined by &&.  Arguments of a wrong type raise what they raise through ctypes. */
static int wrong_type(void)
{
    if (PyErr_ExceptionMatches(PyExc_TypeError)) {
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        PyErr_Format(argument_error, "%S", value ? value : Py_None);
        Py_XDECREF(type);
        Py_XDECREF(value);
        Py_XDECREF(trace);
    }
    return 0;
}
static int integer(PyObject *o, int64_t *out)
{
    *out = PyLong_AsLongLong(o);
    return *out != -1 || !PyErr_Occurred() || wrong_type();
}
static int real(PyObject *o, double *out)
{
    *out = PyFloat_AsDouble(o);
    return *out != -1.0 || !PyErr_Occurred() || wrong_type();
}
/* int32 argument: sizes beyond it are an error, as they are for ctypes' c_int32 callers that check */
static int fits32(int64_t v, int32_t *out)
{
    *out = (int32_t)v;
    if (*out != v) PyErr_Format(PyExc_OverflowError, "%lld does not fit int32", (long long)v);
    return *out == v;
}
static int integer32(PyObject *o, int32_t *out)
{
    int64_t v;
    return integer(o, &v) && fits32(v, out);
}
/* of a method without arguments */
static int ask(PyObject *o, PyObject *method, int64_t *out)
{
    PyObject *r = PyObject_CallMethodNoArgs(o, method);
    if (!r) return 0;
    *out = (int64_t)PyLong_AsUnsignedLongLongMask(r);
    Py_DECREF(r);
    return *out != -1 || !PyErr_Occurred();
}
static int ask32(PyObject *o, PyObject *method, int64_t less, int32_t *out)
{
    int64_t v;
    return ask(o, method, &v) && fits32(v - less, out);
}
/* a tensor's memory, or NULL for None */
static int address(PyObject *o, void **out)
{
    int64_t v = 0;
    const int ok = o == Py_None || ask(o, s_data_ptr, &v);
    *out = (void *)(uintptr_t)v;
    return ok;
}
/* an address as an integer, or NULL for None */
static int pointer(PyObject *o, void **out)
{
    const unsigned long long v = o == Py_None ? 0 : PyLong_AsUnsignedLongLongMask(o);
    *out = (void *)(uintptr_t)v;
    return v != (unsigned long long)-1 || !PyErr_Occurred() || wrong_type();
}
static int stream(void **out)
{
    PyObject *d = PyObject_CallNoArgs(get_device);
    if (!d) return 0;
    PyObject *r = PyObject_CallOneArg(get_stream, d);
    Py_DECREF(d);
    if (!r) return 0;
    const int ok = pointer(r, out);
    Py_DECREF(r);
    return ok;
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

/* None (no buffer) or a tensor */
static int workspace(PyObject *o, void **p, size_t *bytes)
{
    int64_t n = 0, each = 0;
    *p = NULL;
    if (o != Py_None && !(address(o, p) && ask(o, s_numel, &n) && ask(o, s_element_size, &each))) return 0;
    *bytes = (size_t)(n * each);
    return 1;
}

/* spmv(fn, f64, plan, alg, row_ptr, col, val, x, y, alpha, beta, n or None, workspace or None) -> status */
static PyObject *spmv(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    (void)self;
    if (n != 13 || !get_stream) return PyErr_Format(PyExc_TypeError, "spmv: 13 arguments, after streams_from");
    void *fn, *plan, *rp, *col, *val, *x, *y, *ws, *s;
    const int f64 = a[1] == Py_True;
    size_t ws_bytes;
    int32_t m, nnz, cols;
    int64_t alg;
    double alpha, beta;
    if (!(pointer(a[0], &fn) && pointer(a[2], &plan) && integer(a[3], &alg) && ask32(a[4], s_numel, 1, &m) &&
          ask32(a[5], s_numel, 0, &nnz) && (a[11] == Py_None ? ask32(a[7], s_numel, 0, &cols) : integer32(a[11], &cols)) &&
          address(a[4], &rp) && address(a[5], &col) && address(a[6], &val) && address(a[7], &x) && address(a[8], &y) &&
          real(a[9], &alpha) && real(a[10], &beta) && workspace(a[12], &ws, &ws_bytes) && stream(&s)))
        return NULL;
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = f64 ? ((spmv64_t)fn)(plan, (int)alg, m, cols, nnz, alpha, rp, col, val, x, beta, y, ws, ws_bytes, s)
             : ((spmv32_t)fn)(plan, (int)alg, m, cols, nnz, (float)alpha, rp, col, val, x, (float)beta, y, ws, ws_bytes, s);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(st);
}

/* size(d) or stride(d) of a tensor's dimension d */
static int ask_of(PyObject *o, PyObject *method, int64_t d, int64_t *out)
{
    PyObject *i = PyLong_FromLongLong(d);
    PyObject *r = i ? PyObject_CallMethodOneArg(o, method, i) : NULL;
    Py_XDECREF(i);
    if (!r) return 0;
    *out = PyLong_AsLongLong(r);
    Py_DECREF(r);
    return *out != -1 || !PyErr_Occurred();
}
/* Rows of B where the caller does not say: those of ncols elements, ldb apart, that start and end between the tensor's first
 * element and its last.  A view need not hold all that lies between: 8 of 64 columns of 1000 rows are 8000 elements. */
static int rows_of(PyObject *B, int64_t ncols, int64_t ldb, int64_t *rows)
{
    int64_t n, dims, size, stride;
    if (!ask(B, s_numel, &n)) return 0;
    *rows = n / ldb;
    if (n == 0 || ldb == ncols || ldb < 0) return 1;
    if (!ask(B, s_dim, &dims)) return 0;
    int64_t last = 0;
    for (int64_t d = 0; d < dims; ++d) {
        if (!(ask_of(B, s_size, d, &size) && ask_of(B, s_stride, d, &stride))) return 0;
        last += (size - 1) * stride;
    }
    if (last + 1 >= ncols) *rows = (last + 1 - ncols) / ldb + 1;
    return 1;
}

/* spmm(fn, f64, plan, alg, row_ptr, col, val, B, C, ncols, alpha, beta, ldb or None, ldc or None, k or None, workspace or None) -> status */
static PyObject *spmm(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    (void)self;
    if (n != 16 || !get_stream) return PyErr_Format(PyExc_TypeError, "spmm: 16 arguments, after streams_from");
    void *fn, *plan, *rp, *col, *val, *B, *C, *ws, *s;
    const int f64 = a[1] == Py_True;
    size_t ws_bytes;
    int32_t m, nnz, ncols, k;
    int64_t alg, ldb, ldc, rows;
    double alpha, beta;
    if (!(pointer(a[0], &fn) && pointer(a[2], &plan) && integer(a[3], &alg) && ask32(a[4], s_numel, 1, &m) &&
          ask32(a[5], s_numel, 0, &nnz) && integer32(a[9], &ncols)))
        return NULL;
    ldb = ldc = ncols;
    if (!((a[12] == Py_None || integer(a[12], &ldb)) && (a[13] == Py_None || integer(a[13], &ldc)))) return NULL;
    if (a[14] == Py_None && ldb == 0) return PyErr_Format(PyExc_ZeroDivisionError, "spmm: ldb = 0");
    if (!(a[14] == Py_None ? rows_of(a[7], ncols, ldb, &rows) && fits32(rows, &k) : integer32(a[14], &k))) return NULL;
    if (!(address(a[4], &rp) && address(a[5], &col) && address(a[6], &val) && address(a[7], &B) && address(a[8], &C) &&
          real(a[10], &alpha) && real(a[11], &beta) && workspace(a[15], &ws, &ws_bytes) && stream(&s)))
        return NULL;
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = f64 ? ((spmm64_t)fn)(plan, (int)alg, m, k, nnz, ncols, alpha, rp, col, val, B, ldb, beta, C, ldc, ws, ws_bytes, s)
             : ((spmm32_t)fn)(plan, (int)alg, m, k, nnz, ncols, (float)alpha, rp, col, val, B, ldb, (float)beta, C, ldc, ws, ws_bytes, s);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(st);
}

/* plan_values(fn, plan, val) -> status of fn(plan, val, stream) */
static PyObject *plan_values(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    (void)self;
    if (n != 3 || !get_stream) return PyErr_Format(PyExc_TypeError, "plan_values: 3 arguments, after streams_from");
    void *fn, *plan, *val, *s;
    if (!(pointer(a[0], &fn) && pointer(a[1], &plan) && address(a[2], &val) && stream(&s))) return NULL;
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
    s_dim = PyUnicode_InternFromString("dim");
    s_size = PyUnicode_InternFromString("size");
    s_stride = PyUnicode_InternFromString("stride");
    PyObject *ctypes = PyImport_ImportModule("ctypes");
    argument_error = ctypes ? PyObject_GetAttrString(ctypes, "ArgumentError") : NULL;
    Py_XDECREF(ctypes);
    if (!s_data_ptr || !s_numel || !s_element_size || !s_dim || !s_size || !s_stride || !argument_error) return NULL;
    return PyModule_Create(&module);
}
