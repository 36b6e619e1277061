/* Python callables for the entry points that a program calls once per product or attention step.
 *
 * Bound by the caller's own time: such a call is one kernel launch, which takes the HIP runtime 2.5 us, and the generic foreign
 * function interface adds 1.2 us of argument conversion to it.  These callables take plain ints (and a float) straight to the
 * library's function; whatever else they are given -- buffers, None, numpy numbers, too few arguments -- goes to the Python function
 * that they are bound with, which calls through the generic interface, so what is accepted and refused is decided there.
 * matvec_q of Q4_K 4096 x 4096, calls in a row: 4.45 -> 3.97 us.
 *
 * The library is already loaded when the functions are bound, by address: this module links to nothing. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/skainet_hip.h"

typedef int (*matvec_fn)(skn_ctx*, int, const void*, int, int, const float*, float*);
typedef int (*gemm_fn)(skn_ctx*, int, const void*, int, int, const uint16_t*, int, float*);
typedef int (*attn_fn)(skn_ctx*, skn_kv*, const float*, const int32_t*, float, float*);

static matvec_fn matvec_q_at;
static gemm_fn gemm_q_at;
static attn_fn attn_decode_at;
static PyObject *matvec_q_general, *gemm_q_general, *attn_decode_general;

/* true if every one of n arguments is an int of Python's own type */
static int plain(PyObject* const* a, Py_ssize_t n) {
    for (Py_ssize_t i = 0; i < n; i++)
        if (!PyLong_CheckExact(a[i])) return 0;
    return 1;
}
/* as the generic interface converts: modulo the size of the C type */
static void* address(PyObject* o) { return (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(o); }
static int number(PyObject* o) { return (int)PyLong_AsUnsignedLongMask(o); }

static PyObject* matvec_q(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    (void)self;
    if (n != 7 || !plain(a, 7)) return PyObject_Vectorcall(matvec_q_general, a, (size_t)n, NULL);
    skn_ctx* ctx = (skn_ctx*)address(a[0]);
    const int type = number(a[1]), rows = number(a[3]), k = number(a[4]);
    const void* w = address(a[2]);
    const float* x = (const float*)address(a[5]);
    float* y = (float*)address(a[6]);
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = matvec_q_at(ctx, type, w, rows, k, x, y);
    Py_END_ALLOW_THREADS return PyLong_FromLong(rc);
}

static PyObject* gemm_q(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    (void)self;
    if (n != 8 || !plain(a, 8)) return PyObject_Vectorcall(gemm_q_general, a, (size_t)n, NULL);
    skn_ctx* ctx = (skn_ctx*)address(a[0]);
    const int type = number(a[1]), cols = number(a[3]), k = number(a[4]), m = number(a[6]);
    const void* w = address(a[2]);
    const uint16_t* x = (const uint16_t*)address(a[5]);
    float* c = (float*)address(a[7]);
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = gemm_q_at(ctx, type, w, cols, k, x, m, c);
    Py_END_ALLOW_THREADS return PyLong_FromLong(rc);
}

/* (context, cache, q, lengths or None, scale, out) */
static PyObject* attn_decode(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    (void)self;
    if (n != 6 || !plain(a, 3) || a[3] != Py_None || !PyFloat_CheckExact(a[4]) || !plain(a + 5, 1)) return PyObject_Vectorcall(attn_decode_general, a, (size_t)n, NULL);
    skn_ctx* ctx = (skn_ctx*)address(a[0]);
    skn_kv* kv = (skn_kv*)address(a[1]);
    const float* q = (const float*)address(a[2]);
    const float scale = (float)PyFloat_AS_DOUBLE(a[4]);
    float* out = (float*)address(a[5]);
    int rc;
    Py_BEGIN_ALLOW_THREADS rc = attn_decode_at(ctx, kv, q, NULL, scale, out);
    Py_END_ALLOW_THREADS return PyLong_FromLong(rc);
}

/* bind(name, address of the library's function, Python function for other arguments) */
static PyObject* bind(PyObject* self, PyObject* args) {
    const char* name;
    unsigned long long at;
    PyObject* general;
    (void)self;
    if (!PyArg_ParseTuple(args, "sKO", &name, &at, &general)) return NULL;
    PyObject** slot;
    if (!strcmp(name, "matvec_q")) matvec_q_at = (matvec_fn)(uintptr_t)at, slot = &matvec_q_general;
    else if (!strcmp(name, "gemm_q")) gemm_q_at = (gemm_fn)(uintptr_t)at, slot = &gemm_q_general;
    else if (!strcmp(name, "attn_decode")) attn_decode_at = (attn_fn)(uintptr_t)at, slot = &attn_decode_general;
    else return PyErr_Format(PyExc_ValueError, "no entry point %s", name);
    Py_INCREF(general);
    Py_XSETREF(*slot, general);
    Py_RETURN_NONE;
}

static PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, NULL},
                                {"matvec_q", (PyCFunction)(void (*)(void))matvec_q, METH_FASTCALL, NULL},
                                {"gemm_q", (PyCFunction)(void (*)(void))gemm_q, METH_FASTCALL, NULL},
                                {"attn_decode", (PyCFunction)(void (*)(void))attn_decode, METH_FASTCALL, NULL},
                                {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pycall", NULL, -1, methods, NULL, NULL, NULL, NULL};
PyMODINIT_FUNC PyInit__pycall(void) { return PyModule_Create(&module); }
