/* The C ABI's calls of a forward pass as a CPython extension (vectorcall functions): what ctypes converts and looks up for
 * seven to ten arguments takes 0.7 us a call, a third of submitting the launch behind it (quantize + matmul of one token,
 * 2048 x 2048, the first of a burst: 6.6 -> 5.3 us).  Same arguments, conversions and return codes as the ctypes functions of the binding,
 * which stand in where this module is not built; the GIL is released during a call, as there. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/arcz_engine.h"

static PyObject* argument_error; /* ctypes.ArgumentError */

static int bad(PyObject* o) {
  PyErr_Format(argument_error, "argument of type %.100s", Py_TYPE(o)->tp_name);
  return 0;
}
/* an int (as ctypes: any integer, its low 32 bits) */
static int as_int(PyObject* o, int* out) {
  const unsigned long v = PyLong_AsUnsignedLongMask(o);
  if (v == (unsigned long)-1 && PyErr_Occurred()) { PyErr_Clear(); return bad(o); }
  *out = (int)v;
  return 1;
}
/* a handle: an address or None */
static int as_ptr(PyObject* o, void** out) {
  if (o == Py_None) { *out = NULL; return 1; }
  if (!PyLong_Check(o)) return bad(o);
  *out = (void*)(size_t)PyLong_AsUnsignedLongLongMask(o);
  return 1;
}
static int as_float(PyObject* o, float* out) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return bad(o); }
  *out = (float)v;
  return 1;
}
/* arguments by a format of p (handle), i (int), f (float), s (bytes or None) */
union arg { void* p; int i; float f; const char* s; };
static int parse(const char* fmt, PyObject* const* a, Py_ssize_t n, union arg* out) {
  Py_ssize_t k = 0;
  for (; fmt[k]; ++k) {
    if (k >= n) break;
    switch (fmt[k]) {
      case 'p': if (!as_ptr(a[k], &out[k].p)) return 0; break;
      case 'i': if (!as_int(a[k], &out[k].i)) return 0; break;
      case 'f': if (!as_float(a[k], &out[k].f)) return 0; break;
      default:
        if (a[k] == Py_None) out[k].s = NULL;
        else if (PyBytes_Check(a[k])) out[k].s = PyBytes_AS_STRING(a[k]);
        else return bad(a[k]);
    }
  }
  if (fmt[k] || k != n) {
    PyErr_Format(PyExc_TypeError, "this function takes %zd arguments (%zd given)", (Py_ssize_t)strlen(fmt), n);
    return 0;
  }
  return 1;
}
#define CALL(NAME, FMT, EXPR)                                                        \
  static PyObject* NAME(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {  \
    union arg v[12];                                                                 \
    int r;                                                                           \
    (void)self;                                                                      \
    if (!parse(FMT, args, nargs, v)) return NULL;                                    \
    Py_BEGIN_ALLOW_THREADS r = EXPR;                                                 \
    Py_END_ALLOW_THREADS return PyLong_FromLong(r);                                  \
  }
#define E ((arcz_engine*)v[0].p)
CALL(quantize, "ppiiiii", arcz_engine_quantize(E, v[1].p, v[2].i, v[3].i, v[4].i, v[5].i, v[6].i))
CALL(rmsnorm_quant, "ppipiiiifp",
     arcz_engine_rmsnorm_quant(E, v[1].p, v[2].i, v[3].p, v[4].i, v[5].i, v[6].i, v[7].i, v[8].f, v[9].p))
CALL(swiglu_quant, "ppiiiiii", arcz_engine_swiglu_quant(E, v[1].p, v[2].i, v[3].i, v[4].i, v[5].i, v[6].i, v[7].i))
CALL(matmul, "pspipiiii", arcz_engine_matmul(E, v[1].s, v[2].p, v[3].i, v[4].p, v[5].i, v[6].i, v[7].i, v[8].i))
CALL(gemv_gu, "pppip", arcz_engine_gemv_gu(E, v[1].p, v[2].p, v[3].i, v[4].p))
CALL(layer_moe, "pppipii", arcz_engine_layer_moe(E, v[1].p, v[2].p, v[3].i, v[4].p, v[5].i, v[6].i))

#define METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))NAME, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {METHOD(quantize), METHOD(rmsnorm_quant), METHOD(swiglu_quant), METHOD(matmul),
                                METHOD(gemv_gu), METHOD(layer_moe), {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pycall", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__pycall(void) {
  PyObject* ct = PyImport_ImportModule("ctypes");
  if (!ct) return NULL;
  argument_error = PyObject_GetAttrString(ct, "ArgumentError");
  Py_DECREF(ct);
  return argument_error ? PyModule_Create(&module) : NULL;
}
