/* The per-call functions of nart_amd/hipq.py as a CPython extension: tensors in, one call of the hipq C ABI (include/hipq.h).
 *
 * Why: a small operator is one launch, and the launch is 2.6 - 3.2 us of host time in the HIP runtime; through ctypes the way
 * there cost another 1.3 us (three arguments) to 5 us (lists that became numpy arrays and their addresses), so that the
 * eight operators of an inception block took 44 us of host time for 21 us of GPU time.
 *
 * Each function takes the arguments of its namesake in hipq.py, positionally and complete, launches on torch's current stream
 * and returns the C ABI's status.  Nothing of torch is linked: a tensor is asked for data_ptr() and shape. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "hipq.h"

#define MAX_IN HIPQ_MAX_ELTWISE_INPUTS

static PyObject *s_data_ptr, *s_shape, *s_numel;
static PyObject *get_device, *get_stream; /* torch's accessors: () -> int, (int) -> address */

static int current_stream(void **out)
{
    if (get_stream == NULL) {
        PyErr_SetString(PyExc_RuntimeError, "hipq_calls: init() has not been called");
        return 0;
    }
    PyObject *dev = PyObject_CallNoArgs(get_device);
    if (dev == NULL)
        return 0;
    PyObject *st = PyObject_CallOneArg(get_stream, dev);
    Py_DECREF(dev);
    if (st == NULL)
        return 0;
    *out = PyLong_AsVoidPtr(st);
    Py_DECREF(st);
    return !(*out == NULL && PyErr_Occurred());
}

/* a tensor's address; None: a null pointer */
static int address(PyObject *t, void **out)
{
    *out = NULL;
    if (t == Py_None)
        return 1;
    PyObject *v = PyObject_CallMethodNoArgs(t, s_data_ptr);
    if (v == NULL)
        return 0;
    *out = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    return !(*out == NULL && PyErr_Occurred());
}

static int whole(PyObject *o, int *out)
{
    const long v = PyLong_AsLong(o);
    *out = (int)v;
    return !(v == -1 && PyErr_Occurred());
}

static int number(PyObject *o, float *out)
{
    const double v = PyFloat_AsDouble(o);
    *out = (float)v;
    return !(v == -1.0 && PyErr_Occurred());
}

/* the four dimensions of a tensor */
static int shape4(PyObject *t, int d[4])
{
    PyObject *s = PyObject_GetAttr(t, s_shape);
    if (s == NULL)
        return 0;
    int ok = PyTuple_Check(s) && PyTuple_GET_SIZE(s) == 4;
    if (!ok)
        PyErr_SetString(PyExc_ValueError, "a tensor with four dimensions is expected");
    for (int i = 0; ok && i < 4; ++i)
        ok = whole(PyTuple_GET_ITEM(s, i), &d[i]);
    Py_DECREF(s);
    return ok;
}

static int last_dim(PyObject *t, int *out)
{
    PyObject *s = PyObject_GetAttr(t, s_shape);
    if (s == NULL)
        return 0;
    PyObject *v = PySequence_GetItem(s, -1);
    const int ok = v != NULL && whole(v, out);
    Py_XDECREF(v);
    Py_DECREF(s);
    return ok;
}

static int count(PyObject *t, size_t *out)
{
    PyObject *v = PyObject_CallMethodNoArgs(t, s_numel);
    if (v == NULL)
        return 0;
    *out = PyLong_AsSize_t(v);
    Py_DECREF(v);
    return !(*out == (size_t)-1 && PyErr_Occurred());
}

/* the first n entries of a sequence (a list, a tuple, an array) */
static int addresses(PyObject *seq, Py_ssize_t n, const void **out)
{
    for (Py_ssize_t i = 0; i < n; ++i) {
        void *p;
        PyObject *t = PySequence_GetItem(seq, i);
        const int ok = t != NULL && address(t, &p);
        Py_XDECREF(t);
        if (!ok)
            return 0;
        out[i] = p;
    }
    return 1;
}

static int numbers(PyObject *seq, Py_ssize_t n, float *out)
{
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject *v = PySequence_GetItem(seq, i);
        const int ok = v != NULL && number(v, &out[i]);
        Py_XDECREF(v);
        if (!ok)
            return 0;
    }
    return 1;
}

static int wholes(PyObject *seq, Py_ssize_t n, int *out)
{
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject *v = PySequence_GetItem(seq, i);
        const int ok = v != NULL && whole(v, &out[i]);
        Py_XDECREF(v);
        if (!ok)
            return 0;
    }
    return 1;
}

static int bytes_of(PyObject *seq, Py_ssize_t n, uint8_t *out)
{
    int v[MAX_IN];
    if (!wholes(seq, n, v))
        return 0;
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (v[i] < 0 || v[i] > 255) {
            PyErr_SetString(PyExc_OverflowError, "a zero point lies outside 0..255");
            return 0;
        }
        out[i] = (uint8_t)v[i];
    }
    return 1;
}

static int expect(Py_ssize_t got, Py_ssize_t want)
{
    if (got != want)
        PyErr_Format(PyExc_TypeError, "%zd arguments are expected, %zd were given", want, got);
    return got == want;
}

/* a scalar that stands for both directions, or a pair */
static int pair(PyObject *o, int *h, int *w)
{
    if (PyLong_Check(o))
        return whole(o, h) && (*w = *h, 1);
    if (PySequence_Check(o)) {
        const Py_ssize_t n = PySequence_Size(o);
        int v[2];
        if (n != 2) {
            if (n >= 0)
                PyErr_SetString(PyExc_ValueError, "a number or a pair of numbers is expected");
            return 0;
        }
        return wholes(o, 2, v) && (*h = v[0], *w = v[1], 1);
    }
    return whole(o, h) && (*w = *h, 1);
}

#define CALL(EXPR)                         \
    do {                                   \
        int rc_;                           \
        Py_BEGIN_ALLOW_THREADS;            \
        rc_ = (EXPR);                      \
        Py_END_ALLOW_THREADS;              \
        return PyLong_FromLong(rc_);       \
    } while (0)
#define ARGS PyObject *self, PyObject *const *a, Py_ssize_t n

static PyObject *py_init(ARGS)
{
    if (!expect(n, 2))
        return NULL;
    Py_INCREF(a[0]);
    Py_INCREF(a[1]);
    Py_XSETREF(get_device, a[0]);
    Py_XSETREF(get_stream, a[1]);
    Py_RETURN_NONE;
}

/* plan address, x, y, acc */
static PyObject *py_conv2d_run(ARGS)
{
    void *x, *y, *acc, *st;
    if (!expect(n, 4))
        return NULL;
    const void *plan = PyLong_AsVoidPtr(a[0]);
    if ((plan == NULL && PyErr_Occurred()) || !address(a[1], &x) || !address(a[2], &y) || !address(a[3], &acc) || !current_stream(&st))
        return NULL;
    CALL(hipq_conv2d_run((const hipq_conv2d_plan *)plan, x, y, (int32_t *)acc, st));
}

/* a, b, y, ialpha0, izp0, ialpha1, izp1, oalpha, ozp, obits */
static PyObject *py_add_u8(ARGS)
{
    void *p, *q, *y, *st;
    size_t len;
    float a0, a1, ao;
    int z0, z1, zo, bits;
    if (!expect(n, 10) || !address(a[0], &p) || !address(a[1], &q) || !address(a[2], &y) || !count(a[0], &len) || !number(a[3], &a0)
        || !whole(a[4], &z0) || !number(a[5], &a1) || !whole(a[6], &z1) || !number(a[7], &ao) || !whole(a[8], &zo) || !whole(a[9], &bits)
        || !current_stream(&st))
        return NULL;
    CALL(hipq_add_u8(p, q, y, len, a0, z0, a1, z1, ao, zo, bits, st));
}

/* ins, y, ialpha, izp, oalpha, ozp, operation, coeff or None, obits */
static PyObject *py_eltwise_u8(ARGS)
{
    const void *in[MAX_IN];
    float ia[MAX_IN], cf[MAX_IN], ao;
    uint8_t iz[MAX_IN];
    void *y, *st;
    size_t len;
    int zo, op, bits;
    if (!expect(n, 9))
        return NULL;
    const Py_ssize_t m = PySequence_Size(a[0]), k = m < MAX_IN ? m : MAX_IN; /* the C ABI refuses more, by their number */
    if (m < 0 || !addresses(a[0], k, in) || !address(a[1], &y) || !count(a[1], &len) || !numbers(a[2], k, ia) || !bytes_of(a[3], k, iz)
        || !number(a[4], &ao) || !whole(a[5], &zo) || !whole(a[6], &op) || (a[7] != Py_None && !numbers(a[7], k, cf))
        || !whole(a[8], &bits) || !current_stream(&st))
        return NULL;
    CALL(hipq_eltwise_u8(in, (int)m, a[7] == Py_None ? NULL : cf, ia, iz, y, len, op, ao, zo, bits, st));
}

/* x, y, ialpha, izp, oalpha, ozp, obits */
static PyObject *py_relu_u8(ARGS)
{
    void *x, *y, *st;
    size_t len;
    float ai, ao;
    int zi, zo, bits;
    if (!expect(n, 7) || !address(a[0], &x) || !address(a[1], &y) || !count(a[0], &len) || !number(a[2], &ai) || !whole(a[3], &zi)
        || !number(a[4], &ao) || !whole(a[5], &zo) || !whole(a[6], &bits) || !current_stream(&st))
        return NULL;
    CALL(hipq_relu_u8(x, y, len, ai, zi, ao, zo, bits, st));
}

/* ins, channels, y, ialpha, izp, oalpha, ozp, obits */
static PyObject *py_concat_u8(ARGS)
{
    const void *in[MAX_IN];
    float ia[MAX_IN], ao;
    uint8_t iz[MAX_IN];
    int ch[MAX_IN], d[4], zo, bits;
    void *y, *st;
    if (!expect(n, 8))
        return NULL;
    const Py_ssize_t m = PySequence_Size(a[0]), k = m < MAX_IN ? m : MAX_IN; /* the C ABI refuses more, by their number */
    if (m < 0 || !addresses(a[0], k, in) || !wholes(a[1], k, ch) || !address(a[2], &y) || !shape4(a[2], d) || !numbers(a[3], k, ia)
        || !bytes_of(a[4], k, iz) || !number(a[5], &ao) || !whole(a[6], &zo) || !whole(a[7], &bits) || !current_stream(&st))
        return NULL;
    CALL(hipq_concat_u8(in, (int)m, ch, ia, iz, y, (size_t)d[0] * d[1] * d[2], ao, zo, bits, st));
}

/* x, y, C, ialpha, izp, oalpha, ozp, obits */
static PyObject *py_softmax_u8(ARGS)
{
    void *x, *y, *st;
    float ai, ao;
    int d[4], c, zi, zo, bits;
    if (!expect(n, 8) || !address(a[0], &x) || !shape4(a[0], d) || !address(a[1], &y) || !whole(a[2], &c) || !number(a[3], &ai)
        || !whole(a[4], &zi) || !number(a[5], &ao) || !whole(a[6], &zo) || !whole(a[7], &bits) || !current_stream(&st))
        return NULL;
    CALL(hipq_softmax_u8(x, y, (size_t)d[0] * d[1] * d[2], c, d[3], ai, zi, ao, zo, bits, st));
}

/* x, y, C, kernel, pad, stride, method, ialpha, izp, oalpha, ozp, obits */
static PyObject *py_pool_u8(ARGS)
{
    void *x, *y, *st;
    float ai, ao;
    int d[4], o[4], c, kh, kw, ph, pw, sh, sw, method, zi, zo, bits;
    if (!expect(n, 12) || !address(a[0], &x) || !shape4(a[0], d) || !address(a[1], &y) || !shape4(a[1], o) || !whole(a[2], &c)
        || !pair(a[3], &kh, &kw) || !pair(a[4], &ph, &pw) || !pair(a[5], &sh, &sw) || !whole(a[6], &method) || !number(a[7], &ai)
        || !whole(a[8], &zi) || !number(a[9], &ao) || !whole(a[10], &zo) || !whole(a[11], &bits) || !current_stream(&st))
        return NULL;
    CALL(hipq_pool_u8(x, y, d[0], c, d[1], d[2], o[1], o[2], d[3], kh, kw, ph, pw, sh, sw, method, ai, zi, ao, zo, bits, st));
}

/* x (NCHW floats), y (NHWC bytes), oalpha, ozp, obits */
static PyObject *py_quantize_u8(ARGS)
{
    void *x, *y, *st;
    float ao;
    int d[4], cs, zo, bits;
    if (!expect(n, 5) || !address(a[0], &x) || !shape4(a[0], d) || !address(a[1], &y) || !last_dim(a[1], &cs) || !number(a[2], &ao)
        || !whole(a[3], &zo) || !whole(a[4], &bits) || !current_stream(&st))
        return NULL;
    CALL(hipq_quantize_u8(x, y, d[0], d[1], d[2], d[3], cs, ao, zo, bits, st));
}

/* x (NCHW floats), y (NHWC bytes), oalpha, obits */
static PyObject *py_quantize_i8(ARGS)
{
    void *x, *y, *st;
    float ao;
    int d[4], cs, bits;
    if (!expect(n, 4) || !address(a[0], &x) || !shape4(a[0], d) || !address(a[1], &y) || !last_dim(a[1], &cs) || !number(a[2], &ao)
        || !whole(a[3], &bits) || !current_stream(&st))
        return NULL;
    CALL(hipq_quantize_i8(x, y, d[0], d[1], d[2], d[3], cs, ao, bits, st));
}

/* x (NHWC bytes), y (NCHW floats), ialpha, izp */
static PyObject *py_dequantize_u8(ARGS)
{
    void *x, *y, *st;
    float ai;
    int cs, o[4], zi;
    if (!expect(n, 4) || !address(a[0], &x) || !last_dim(a[0], &cs) || !address(a[1], &y) || !shape4(a[1], o) || !number(a[2], &ai)
        || !whole(a[3], &zi) || !current_stream(&st))
        return NULL;
    CALL(hipq_dequantize_u8(x, y, o[0], o[1], o[2], o[3], cs, ai, zi, st));
}

/* x (NHWC bytes), y (NCHW floats), ialpha */
static PyObject *py_dequantize_i8(ARGS)
{
    void *x, *y, *st;
    float ai;
    int cs, o[4];
    if (!expect(n, 3) || !address(a[0], &x) || !last_dim(a[0], &cs) || !address(a[1], &y) || !shape4(a[1], o) || !number(a[2], &ai)
        || !current_stream(&st))
        return NULL;
    CALL(hipq_dequantize_i8(x, y, o[0], o[1], o[2], o[3], cs, ai, st));
}

#define METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))py_##NAME, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {
    METHOD(init),        METHOD(conv2d_run),  METHOD(add_u8),      METHOD(eltwise_u8),    METHOD(relu_u8),       METHOD(concat_u8), METHOD(softmax_u8),
    METHOD(pool_u8),     METHOD(quantize_u8), METHOD(quantize_i8), METHOD(dequantize_u8), METHOD(dequantize_i8), {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "hipq_calls", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit_hipq_calls(void)
{
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_shape = PyUnicode_InternFromString("shape");
    s_numel = PyUnicode_InternFromString("numel");
    return s_data_ptr && s_shape && s_numel ? PyModule_Create(&module) : NULL;
}
