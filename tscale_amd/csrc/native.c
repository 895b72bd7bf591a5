/* The Python side's calls into the library (CPython extension, no framework headers): a Call object fills an argument struct
 * of include/tsattn.h from positional values and calls the entry point, without a ctypes structure per call (30 to 50
 * attribute writes of 0.1 to 0.2 us each, which is more than a small launch takes on the GPU).  A pointer value may be None,
 * an integer address, bytes (what Call.pack() made: a struct inside a struct) or anything with a data_ptr() method. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/tsattn.h"

static PyObject *s_data_ptr; /* "data_ptr" */

static int as_pointer(PyObject *v, void **out)
{
    if (v == Py_None) {
        *out = NULL;
        return 0;
    }
    if (PyLong_CheckExact(v)) {
        *out = PyLong_AsVoidPtr(v);
        return *out == NULL && PyErr_Occurred() ? -1 : 0;
    }
    if (PyBytes_CheckExact(v)) {
        *out = PyBytes_AS_STRING(v);
        return 0;
    }
    PyObject *r = PyObject_CallMethodNoArgs(v, s_data_ptr);
    if (!r) return -1;
    *out = PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    return *out == NULL && PyErr_Occurred() ? -1 : 0;
}

/* ---- Call(address, size, fields): fields = bytes of (offset u16, kind u8) triples, kind one of "iqfp" ------------------- */
#define MAX_FIELDS 64
#define MAX_STRUCT 1024
typedef struct {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    int (*fn)(void *, const void *, void *);
    int size, n_fields;
    uint16_t offset[MAX_FIELDS];
    char kind[MAX_FIELDS];
} Call;

static int fill(const Call *c, char *at, PyObject *const *values, Py_ssize_t n)
{
    if (n > c->n_fields) {
        PyErr_SetString(PyExc_TypeError, "more values than the struct has fields");
        return -1;
    }
    memset(at, 0, (size_t)c->size);
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject *const v = values[i];
        char *const dst = at + c->offset[i];
        switch (c->kind[i]) {
        case 'p': {
            void *p;
            if (as_pointer(v, &p)) return -1;
            memcpy(dst, &p, sizeof p);
            break;
        }
        case 'f': {
            const double d = PyFloat_AsDouble(v);
            if (d == -1.0 && PyErr_Occurred()) return -1;
            const float f = (float)d;
            memcpy(dst, &f, sizeof f);
            break;
        }
        default: {
            const long long x = PyLong_AsLongLong(v);
            if (x == -1 && PyErr_Occurred()) return -1;
            if (c->kind[i] == 'q') {
                const int64_t q = x;
                memcpy(dst, &q, sizeof q);
            } else {
                if (x < INT32_MIN || x > INT32_MAX) {
                    PyErr_Format(PyExc_OverflowError, "value %lld does not fit an int field", x);
                    return -1;
                }
                const int32_t q = (int32_t)x;
                memcpy(dst, &q, sizeof q);
            }
        }
        }
    }
    return 0;
}

/* call(handle, stream, value, ...): values in the order of the fields, the rest zero; returns the status */
static PyObject *call_vectorcall(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kw)
{
    Call *const c = (Call *)self;
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    if (n < 2 || (kw && PyTuple_GET_SIZE(kw))) {
        PyErr_SetString(PyExc_TypeError, "call(handle, stream, value, ...)");
        return NULL;
    }
    void *handle, *stream;
    if (as_pointer(args[0], &handle) || as_pointer(args[1], &stream)) return NULL;
    uint64_t mem[MAX_STRUCT / 8];
    if (fill(c, (char *)mem, args + 2, n - 2)) return NULL;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = c->fn(handle, mem, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

/* call.pack(value, ...): the struct as bytes, for a pointer field of another call */
static PyObject *call_pack(PyObject *self, PyObject *const *args, Py_ssize_t n)
{
    Call *const c = (Call *)self;
    PyObject *const b = PyBytes_FromStringAndSize(NULL, c->size);
    if (!b) return NULL;
    if (fill(c, PyBytes_AS_STRING(b), args, n)) {
        Py_DECREF(b);
        return NULL;
    }
    return b;
}

static PyMethodDef call_methods[] = {
    {"pack", (PyCFunction)(void (*)(void))call_pack, METH_FASTCALL, "the struct as bytes"},
    {NULL, NULL, 0, NULL},
};

static PyObject *call_new(PyTypeObject *type, PyObject *args, PyObject *kw)
{
    (void)kw;
    unsigned long long address;
    int size;
    const unsigned char *f;
    Py_ssize_t len;
    if (!PyArg_ParseTuple(args, "Kiy#", &address, &size, &f, &len)) return NULL;
    if (size <= 0 || size > MAX_STRUCT || len % 3 || len / 3 > MAX_FIELDS) {
        PyErr_SetString(PyExc_ValueError, "struct or field list too large");
        return NULL;
    }
    Call *const c = (Call *)type->tp_alloc(type, 0);
    if (!c) return NULL;
    c->vectorcall = call_vectorcall;
    c->fn = (int (*)(void *, const void *, void *))(uintptr_t)address;
    c->size = size;
    c->n_fields = (int)(len / 3);
    for (int i = 0; i < c->n_fields; ++i) {
        c->offset[i] = (uint16_t)(f[3 * i] | f[3 * i + 1] << 8);
        c->kind[i] = (char)f[3 * i + 2];
        const int bytes = c->kind[i] == 'i' || c->kind[i] == 'f' ? 4 : 8;
        if (c->offset[i] + bytes > size) {
            Py_DECREF(c);
            PyErr_SetString(PyExc_ValueError, "field outside the struct");
            return NULL;
        }
    }
    return (PyObject *)c;
}

static PyTypeObject CallType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "tscale_amd._native.Call",
    .tp_basicsize = sizeof(Call),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL,
    .tp_vectorcall_offset = offsetof(Call, vectorcall),
    .tp_call = PyVectorcall_Call,
    .tp_methods = call_methods,
    .tp_new = call_new,
};

/* ---- entry points that take their arguments one by one; addresses from bind() ------------------------------------------ */
typedef union {
    void *p;
    int64_t q;
    double f;
} Value;

static int parse(const char *kinds, PyObject *const *args, Py_ssize_t n, Value *v)
{
    if (n != (Py_ssize_t)strlen(kinds)) {
        PyErr_Format(PyExc_TypeError, "%zd arguments wanted, %zd given", (Py_ssize_t)strlen(kinds), n);
        return -1;
    }
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (kinds[i] == 'p') {
            if (as_pointer(args[i], &v[i].p)) return -1;
        } else if (kinds[i] == 'f') {
            v[i].f = PyFloat_AsDouble(args[i]);
            if (v[i].f == -1.0 && PyErr_Occurred()) return -1;
        } else if (kinds[i] == 'u') {
            v[i].q = (int64_t)PyLong_AsUnsignedLongLongMask(args[i]);
            if (v[i].q == -1 && PyErr_Occurred()) return -1;
        } else {
            v[i].q = PyLong_AsLongLong(args[i]);
            if (v[i].q == -1 && PyErr_Occurred()) return -1;
            if (kinds[i] == 'i' && (v[i].q < INT32_MIN || v[i].q > INT32_MAX)) {
                PyErr_Format(PyExc_OverflowError, "argument %zd does not fit an int", i);
                return -1;
            }
        }
    }
    return 0;
}

static struct {
    __typeof__(tsattn_quantize_rows) *quantize_rows;
    __typeof__(tsattn_build_spans) *build_spans;
    __typeof__(tsattn_build_span_tiles) *build_span_tiles;
    __typeof__(tsattn_embed_rows) *embed_rows;
    __typeof__(tsattn_softmax_rows_scratch) *softmax_rows;
    __typeof__(tsattn_sample_rows_scratch) *sample_rows;
    __typeof__(tsattn_kv_product) *kv_product;
} lib;

static PyObject *bind(PyObject *self, PyObject *args)
{
    (void)self;
    unsigned long long a[7];
    if (!PyArg_ParseTuple(args, "KKKKKKK", a, a + 1, a + 2, a + 3, a + 4, a + 5, a + 6)) return NULL;
    lib.quantize_rows = (__typeof__(lib.quantize_rows))(uintptr_t)a[0];
    lib.build_spans = (__typeof__(lib.build_spans))(uintptr_t)a[1];
    lib.build_span_tiles = (__typeof__(lib.build_span_tiles))(uintptr_t)a[2];
    lib.embed_rows = (__typeof__(lib.embed_rows))(uintptr_t)a[3];
    lib.softmax_rows = (__typeof__(lib.softmax_rows))(uintptr_t)a[4];
    lib.sample_rows = (__typeof__(lib.sample_rows))(uintptr_t)a[5];
    lib.kv_product = (__typeof__(lib.kv_product))(uintptr_t)a[6];
    Py_RETURN_NONE;
}

#define FLAT(name, kinds, ...)                                                                 \
    static PyObject *name(PyObject *self, PyObject *const *args, Py_ssize_t n)                 \
    {                                                                                          \
        (void)self;                                                                            \
        Value v[sizeof(kinds)];                                                                \
        if (!lib.name) {                                                                       \
            PyErr_SetString(PyExc_RuntimeError, "the library has not been bound");             \
            return NULL;                                                                       \
        }                                                                                      \
        if (parse(kinds, args, n, v)) return NULL;                                             \
        int rc;                                                                                \
        Py_BEGIN_ALLOW_THREADS rc = lib.name(__VA_ARGS__);                                     \
        Py_END_ALLOW_THREADS return PyLong_FromLong(rc);                                       \
    }
#define I(k) (int)v[k].q
#define F(k) (float)v[k].f
FLAT(quantize_rows, "piipqqiipqpqp", v[0].p, I(1), I(2), v[3].p, v[4].q, v[5].q, I(6), I(7), v[8].p, v[9].q, v[10].p, v[11].q, v[12].p)
FLAT(build_spans, "pipqpqppp", v[0].p, I(1), v[2].p, v[3].q, v[4].p, v[5].q, v[6].p, v[7].p, v[8].p)
FLAT(build_span_tiles, "pqpppp", v[0].p, v[1].q, v[2].p, v[3].p, v[4].p, v[5].p)
FLAT(embed_rows, "pqipipqqfpqp", v[0].p, v[1].q, I(2), v[3].p, I(4), v[5].p, v[6].q, v[7].q, F(8), v[9].p, v[10].q, v[11].p)
FLAT(softmax_rows, "pqqpiqqfppqppqp", v[0].p, v[1].q, v[2].q, v[3].p, I(4), v[5].q, v[6].q, F(7), v[8].p, v[9].p, v[10].q, v[11].p, v[12].p, v[13].q, v[14].p)
FLAT(sample_rows, "pqqpqfpquuppqp", v[0].p, v[1].q, v[2].q, v[3].p, v[4].q, F(5), v[6].p, v[7].q, (uint64_t)v[8].q, (uint64_t)v[9].q, v[10].p, v[11].p, v[12].q, v[13].p)
FLAT(kv_product, "pqiiipqipqfpqp", v[0].p, v[1].q, I(2), I(3), I(4), v[5].p, v[6].q, I(7), v[8].p, v[9].q, F(10), v[11].p, v[12].q, v[13].p)

static PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "addresses of the functions below"},
    {"quantize_rows", (PyCFunction)(void (*)(void))quantize_rows, METH_FASTCALL, NULL},
    {"build_spans", (PyCFunction)(void (*)(void))build_spans, METH_FASTCALL, NULL},
    {"build_span_tiles", (PyCFunction)(void (*)(void))build_span_tiles, METH_FASTCALL, NULL},
    {"embed_rows", (PyCFunction)(void (*)(void))embed_rows, METH_FASTCALL, NULL},
    {"softmax_rows", (PyCFunction)(void (*)(void))softmax_rows, METH_FASTCALL, NULL},
    {"sample_rows", (PyCFunction)(void (*)(void))sample_rows, METH_FASTCALL, NULL},
    {"kv_product", (PyCFunction)(void (*)(void))kv_product, METH_FASTCALL, NULL},
    {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__native(void)
{
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    if (!s_data_ptr || PyType_Ready(&CallType) < 0) return NULL;
    PyObject *const m = PyModule_Create(&module);
    if (!m) return NULL;
    Py_INCREF(&CallType);
    if (PyModule_AddObject(m, "Call", (PyObject *)&CallType) < 0) return NULL;
    return m;
}
