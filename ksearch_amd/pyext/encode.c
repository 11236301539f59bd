/* The one call of the binding that a caller's own loop makes per operator: ksh_encode, without ctypes in between.
 *
 * Appending a launch takes the library about 2.5 us (almost all of it in the HIP runtime); building four ctypes arrays
 * and converting eight arguments took 3 us more, so a 4096 x 4096 GEMV (3.6 us on the GPU) was issued every 6.4 us.
 * Here the handles and offsets go straight from the Python sequences into C arrays.
 *
 *   setup(address of ksh_encode)
 *   encode(ctx, kernel, inputs, in_offs, outputs, out_offs) -> the library's return code
 * ctx and kernel are integers; inputs / outputs are iterables of objects with a handle in attribute `h` (None: a null
 * binding, which the library refuses); offsets are None or iterables of byte offsets, taken as int() takes them.  The
 * ctypes form of the same call (hip.py, _encode_ctypes) accepts and refuses what this one does.
 *
 * Built against the limited API: one binary for every CPython from 3.10 on. */
#define PY_SSIZE_T_CLEAN
#define Py_LIMITED_API 0x030a0000
#include <Python.h>
#include <stdint.h>

enum { kMax = 16 }; /* more bindings than any kernel has; the library checks the exact number */

typedef int (*encode_fn)(void *, void *, void *const *, const uint64_t *, int, void *const *, const uint64_t *, int);
static encode_fn g_encode;
static PyObject *g_h;

static int as_ptr(PyObject *o, void **out)
{
    if (o == Py_None) { *out = NULL; return 0; }
    *out = PyLong_AsVoidPtr(o);
    return PyErr_Occurred() ? -1 : 0;
}

/* item i (borrowed) of what PySequence_Fast returned */
static PyObject *item(PyObject *seq, int is_list, Py_ssize_t i) { return is_list ? PyList_GetItem(seq, i) : PyTuple_GetItem(seq, i); }

/* handles of a sequence of buffers, and their offsets (zero where there are none); of more than any kernel has only the
 * number, which the library refuses before it looks at them */
static int bindings(PyObject *bufs, PyObject *offs, void **ptr, uint64_t *off)
{
    PyObject *b = PySequence_Fast(bufs, "bindings are an iterable of buffers"), *o = NULL;
    if (!b) return -1;
    const int b_list = PyList_Check(b);
    const Py_ssize_t n = PySequence_Size(b);
    Py_ssize_t n_off = 0;
    int rc = -1, o_list = 0;
    if (offs != Py_None) {
        o = PySequence_Fast(offs, "offsets are an iterable of numbers");
        if (!o) goto done;
        o_list = PyList_Check(o);
        n_off = PySequence_Size(o);
        if (n_off > (n ? n : 1)) {
            PyErr_SetString(PyExc_IndexError, "more offsets than bindings");
            goto done;
        }
    }
    for (Py_ssize_t i = 0; i < n && i < kMax; i++) {
        PyObject *e = item(b, b_list, i), *h = e ? PyObject_GetAttr(e, g_h) : NULL;
        if (!h) goto done;
        const int bad = as_ptr(h, &ptr[i]);
        Py_DECREF(h);
        if (bad) goto done;
        off[i] = 0;
        if (i < n_off) {
            PyObject *e_off = item(o, o_list, i), *v = e_off ? PyNumber_Long(e_off) : NULL;
            if (!v) goto done;
            off[i] = PyLong_AsUnsignedLongLongMask(v);
            Py_DECREF(v);
        }
    }
    rc = (int)n;
done:
    Py_DECREF(b);
    Py_XDECREF(o);
    return rc;
}

static PyObject *encode(PyObject *self, PyObject *const *args, Py_ssize_t nargs)
{
    void *ctx, *kernel, *in[kMax], *out[kMax];
    uint64_t in_off[kMax], out_off[kMax];
    int n_in, n_out, rc;
    (void)self;
    if (nargs != 6 || !g_encode) {
        PyErr_SetString(PyExc_TypeError, "encode(ctx, kernel, inputs, in_offs, outputs, out_offs) after setup()");
        return NULL;
    }
    if (as_ptr(args[0], &ctx) || as_ptr(args[1], &kernel)) return NULL;
    if ((n_in = bindings(args[2], args[3], in, in_off)) < 0 || (n_out = bindings(args[4], args[5], out, out_off)) < 0) return NULL;
    Py_BEGIN_ALLOW_THREADS
    rc = g_encode(ctx, kernel, in, in_off, n_in, out, out_off, n_out);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

static PyObject *setup(PyObject *self, PyObject *addr)
{
    void *p;
    (void)self;
    if (as_ptr(addr, &p)) return NULL;
    g_encode = (encode_fn)(uintptr_t)p;
    Py_RETURN_NONE;
}

static PyMethodDef methods[] = {
    {"encode", (PyCFunction)(void (*)(void))encode, METH_FASTCALL, "append one launch; returns ksh_encode's code"},
    {"setup", setup, METH_O, "the address of ksh_encode"},
    {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_encode", "ksh_encode without ctypes", -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__encode(void)
{
    g_h = PyUnicode_InternFromString("h");
    return g_h ? PyModule_Create(&module) : NULL;
}
