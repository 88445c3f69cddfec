/* The launch path of caminus_amd.device.hip and caminus_amd.engine.k3 without ctypes: a decode step is a few launches of small kernels, and
 * building a ctypes object per argument and converting it again cost their caller 1.2 to 3.1 us a launch beside the 3.8 us in hipLaunchKernel.
 * With it, a decode token's row ops (4 launches) go from 24.3 to 18.7 us, a verify pass of 4 tokens (5 launches) from
 * 33.2 to 26.5 and a batch of 48 sequences (3 launches) from 22.0 to 18.2; hipLaunchKernel itself and then the kernels bound what is left.
 *
 *   bind(address, signature) -> entry; entry(*args) -> the C function's int. One character per argument: 'p' a tensor's data pointer or None, 'a'
 *       an integer address, 'i' / 'l' an int / long (any object with __index__, reduced to its width as ctypes reduces it), 'f' a float. Any other
 *       type is a TypeError and nothing is called.
 *   call(address, *args) -> the same for arguments that carry their type, a torch.Tensor, None or a ctypes c_int / c_long / c_float / c_void_p
 *       instance; NotImplemented, with nothing called, for anything else.
 *   setup(Tensor, c_int, c_long, c_float, c_void_p): the types call() looks for.
 *
 * The C entry points take pointers, ints, longs and floats only. In the x86-64 calling convention the first six integer arguments and the
 * first eight floats travel in registers of their own kind whatever their order, and further integers on the stack in order, each in
 * eight bytes: so one prototype with the integers and floats of a call listed apart fits every entry point, arguments it does not have included. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stddef.h>
#if !defined(__x86_64__)
#error "the calling convention above is x86-64's"
#endif
#define MAX_INTS 40
#define MAX_FLOATS 8
typedef long L;
typedef int (*any_fn)(L, L, L, L, L, L, float, float, float, float, float, float, float, float, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L, L,
                      L, L, L, L, L, L);
typedef struct { L i[MAX_INTS]; float f[MAX_FLOATS]; int ni, nf; } Args;

static PyObject * t_tensor, * t_int, * t_long, * t_float, * t_ptr, * s_data_ptr, * s_value;

static PyObject * go(void * fn, const Args * a) {
    int rc;
    const L * i = a->i; const float * f = a->f;
    Py_BEGIN_ALLOW_THREADS
    if (a->ni <= 16)
        rc = ((int (*)(L, L, L, L, L, L, float, float, float, float, float, float, float, float, L, L, L, L, L, L, L, L, L, L))fn)(
            i[0], i[1], i[2], i[3], i[4], i[5], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7], i[6], i[7], i[8], i[9], i[10], i[11], i[12], i[13], i[14], i[15]);
    else
        rc = ((any_fn)fn)(i[0], i[1], i[2], i[3], i[4], i[5], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7], i[6], i[7], i[8], i[9], i[10], i[11], i[12], i[13], i[14], i[15],
                          i[16], i[17], i[18], i[19], i[20], i[21], i[22], i[23], i[24], i[25], i[26], i[27], i[28], i[29], i[30], i[31], i[32], i[33], i[34], i[35], i[36], i[37],
                          i[38], i[39]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}
/* an object's address: a tensor's data pointer */
static int data_pointer(PyObject * o, L * out) {
    PyObject * v = PyObject_CallMethodNoArgs(o, s_data_ptr);
    if (!v) return -1;
    *out = (L)PyLong_AsUnsignedLongMask(v);
    Py_DECREF(v);
    return PyErr_Occurred() ? -1 : 0;
}
static int integer(PyObject * o, int is_long, L * out) {
    PyObject * v = PyLong_CheckExact(o) ? (Py_INCREF(o), o) : PyNumber_Index(o);
    if (!v) return -1;
    const unsigned long u = PyLong_AsUnsignedLongMask(v);
    Py_DECREF(v);
    if (PyErr_Occurred()) return -1;
    *out = is_long ? (L)u : (L)(int)u;
    return 0;
}

typedef struct { PyObject_HEAD vectorcallfunc vectorcall; void * fn; int n; char sig[MAX_INTS + MAX_FLOATS + 1]; } Entry;
static PyObject * entry_call(PyObject * self, PyObject * const * args, size_t nargsf, PyObject * kw) {
    Entry * e = (Entry *)self;
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    if (n != e->n || (kw && PyTuple_GET_SIZE(kw))) { PyErr_Format(PyExc_TypeError, "this entry point takes %d positional arguments (%zd given)", e->n, n); return NULL; }
    Args a;
    a.ni = a.nf = 0;
    for (int k = 0; k < n; k++) {
        PyObject * o = args[k];
        switch (e->sig[k]) {
        case 'p':
            if (o == Py_None) a.i[a.ni++] = 0;
            else if (data_pointer(o, &a.i[a.ni++])) return NULL;
            break;
        case 'i': if (integer(o, 0, &a.i[a.ni++])) return NULL; break;
        case 'l': case 'a': if (integer(o, 1, &a.i[a.ni++])) return NULL; break;
        default: {
            const double d = PyFloat_AsDouble(o);
            if (d == -1.0 && PyErr_Occurred()) return NULL;
            a.f[a.nf++] = (float)d;
        }
        }
    }
    for (int k = a.ni; k < (a.ni <= 16 ? 16 : MAX_INTS); k++) a.i[k] = 0;
    for (int k = a.nf; k < MAX_FLOATS; k++) a.f[k] = 0.0f;
    return go(e->fn, &a);
}
static PyTypeObject EntryType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "caminus_amd.device._launch.Entry", .tp_basicsize = sizeof(Entry), .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL,
    .tp_vectorcall_offset = offsetof(Entry, vectorcall), .tp_call = PyVectorcall_Call,
};
static PyObject * bind(PyObject * self, PyObject * args) {
    PyObject * addr; const char * sig; Py_ssize_t len;
    (void)self;
    if (!PyArg_ParseTuple(args, "Os#", &addr, &sig, &len)) return NULL;
    int ni = 0, nf = 0;
    for (Py_ssize_t k = 0; k < len; k++) {
        if (!memchr("pailf", sig[k], 5)) { PyErr_Format(PyExc_ValueError, "signature %s: one of p, a, i, l, f per argument", sig); return NULL; }
        if (sig[k] == 'f') nf++; else ni++;
    }
    if (ni > MAX_INTS || nf > MAX_FLOATS) { PyErr_Format(PyExc_ValueError, "signature %s: at most %d integers and %d floats", sig, MAX_INTS, MAX_FLOATS); return NULL; }
    void * fn = PyLong_AsVoidPtr(addr);
    if (!fn) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point"); return NULL; }
    Entry * e = PyObject_New(Entry, &EntryType);
    if (!e) return NULL;
    e->vectorcall = entry_call; e->fn = fn; e->n = (int)len;
    memcpy(e->sig, sig, (size_t)len + 1);
    return (PyObject *)e;
}
static PyObject * call(PyObject * self, PyObject * const * args, Py_ssize_t n) {
    (void)self;
    if (!t_tensor || n < 1) { PyErr_SetString(PyExc_RuntimeError, "call(address, ..) after setup(..)"); return NULL; }
    void * fn = PyLong_AsVoidPtr(args[0]);
    if (!fn) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point"); return NULL; }
    Args a;
    a.ni = a.nf = 0;
    for (Py_ssize_t k = 1; k < n; k++) {
        PyObject * o = args[k], * t = (PyObject *)Py_TYPE(o);
        if ((t == t_float ? a.nf >= MAX_FLOATS : a.ni >= MAX_INTS)) Py_RETURN_NOTIMPLEMENTED;
        if (t == t_tensor) { if (data_pointer(o, &a.i[a.ni++])) return NULL; continue; }
        if (o == Py_None) { a.i[a.ni++] = 0; continue; }
        if (t != t_int && t != t_long && t != t_float && t != t_ptr) Py_RETURN_NOTIMPLEMENTED;
        PyObject * v = PyObject_GetAttr(o, s_value);
        if (!v) return NULL;
        if (t == t_float) a.f[a.nf++] = (float)PyFloat_AsDouble(v);
        else if (v == Py_None) a.i[a.ni++] = 0;
        else if (integer(v, t != t_int, &a.i[a.ni++])) { Py_DECREF(v); return NULL; }
        Py_DECREF(v);
        if (PyErr_Occurred()) return NULL;
    }
    for (int k = a.ni; k < (a.ni <= 16 ? 16 : MAX_INTS); k++) a.i[k] = 0;
    for (int k = a.nf; k < MAX_FLOATS; k++) a.f[k] = 0.0f;
    return go(fn, &a);
}
static PyObject * setup(PyObject * self, PyObject * args) {
    PyObject * a, * b, * c, * d, * e;
    (void)self;
    if (!PyArg_ParseTuple(args, "OOOOO", &a, &b, &c, &d, &e)) return NULL;
    Py_XINCREF(a); Py_XINCREF(b); Py_XINCREF(c); Py_XINCREF(d); Py_XINCREF(e);
    t_tensor = a; t_int = b; t_long = c; t_float = d; t_ptr = e;
    Py_RETURN_NONE;
}
static PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "bind(address, signature) -> entry"},
    {"call", (PyCFunction)(void (*)(void))call, METH_FASTCALL, "call(address, *typed arguments) -> int or NotImplemented"},
    {"setup", setup, METH_VARARGS, "setup(Tensor, c_int, c_long, c_float, c_void_p)"},
    {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", "launches without ctypes", -1, methods, NULL, NULL, NULL, NULL};
PyMODINIT_FUNC PyInit__launch(void) {
    if (PyType_Ready(&EntryType) < 0) return NULL;
    s_data_ptr = PyUnicode_InternFromString("data_ptr"); s_value = PyUnicode_InternFromString("value");
    return s_data_ptr && s_value ? PyModule_Create(&module) : NULL;
}
