/* The C ABI's calls of a forward pass as a CPython extension (vectorcall functions): what ctypes converts and looks up for
 * seven to ten arguments takes 0.7 us a call, a third of submitting the launch behind it (quantize + matmul of one token,
 * 2048 x 2048, the first of a burst: 6.6 -> 5.3 us).  Plain arguments -- int, float, bytes, None as they come -- are converted here;
 * a call with any other, or with another number of them, goes to the ctypes function of the binding as it is (bind), which
 * takes or refuses it.  The GIL is released during a call, as there. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/arcz_engine.h"

/* arguments by a format of p (handle), i (int), f (float), s (bytes or None) */
union arg { void* p; int i; float f; const char* s; };
static int plain(const char* fmt, PyObject* const* a, Py_ssize_t n, union arg* out) {
  Py_ssize_t k = 0;
  for (; fmt[k] && k < n; ++k) {
    PyObject* o = a[k];
    if (fmt[k] == 'f') {
      if (!PyFloat_CheckExact(o)) return 0;
      out[k].f = (float)PyFloat_AS_DOUBLE(o);
    } else if (fmt[k] == 'i') {  /* (its low 32 bits) */
      if (!PyLong_Check(o)) return 0;
      out[k].i = (int)PyLong_AsUnsignedLongMask(o);
    } else if (o == Py_None) {
      out[k].p = NULL;
    } else if (fmt[k] == 's') {
      if (!PyBytes_CheckExact(o)) return 0;
      out[k].s = PyBytes_AS_STRING(o);
    } else {
      if (!PyLong_Check(o)) return 0;
      out[k].p = (void*)PyLong_AsUnsignedLongMask(o);
    }
  }
  return !fmt[k] && k == n;
}
#define CALL(NAME, FMT, EXPR)                                                        \
  static PyObject* NAME##_ctypes;                                                    \
  static PyObject* NAME(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {  \
    union arg v[12];                                                                 \
    int r;                                                                           \
    (void)self;                                                                      \
    if (!plain(FMT, args, nargs, v)) return otherwise(NAME##_ctypes, args, nargs);   \
    Py_BEGIN_ALLOW_THREADS r = EXPR;                                                 \
    Py_END_ALLOW_THREADS return PyLong_FromLong(r);                                  \
  }
static PyObject* otherwise(PyObject* f, PyObject* const* args, Py_ssize_t nargs) {
  if (f) return PyObject_Vectorcall(f, args, (size_t)nargs, NULL);
  PyErr_SetString(PyExc_TypeError, "arguments for the ctypes function, and none is bound");
  return NULL;
}
#define E ((arcz_engine*)v[0].p)
CALL(quantize, "ppiiiii", arcz_engine_quantize(E, v[1].p, v[2].i, v[3].i, v[4].i, v[5].i, v[6].i))
CALL(rmsnorm_quant, "ppipiiiifp",
     arcz_engine_rmsnorm_quant(E, v[1].p, v[2].i, v[3].p, v[4].i, v[5].i, v[6].i, v[7].i, v[8].f, v[9].p))
CALL(swiglu_quant, "ppiiiiii", arcz_engine_swiglu_quant(E, v[1].p, v[2].i, v[3].i, v[4].i, v[5].i, v[6].i, v[7].i))
CALL(matmul, "pspipiiii", arcz_engine_matmul(E, v[1].s, v[2].p, v[3].i, v[4].p, v[5].i, v[6].i, v[7].i, v[8].i))
CALL(gemv_gu, "pppip", arcz_engine_gemv_gu(E, v[1].p, v[2].p, v[3].i, v[4].p))
CALL(layer_moe, "pppipii", arcz_engine_layer_moe(E, v[1].p, v[2].p, v[3].i, v[4].p, v[5].i, v[6].i))

/* bind(quantize, rmsnorm_quant, swiglu_quant, matmul, gemv_gu, layer_moe): the ctypes functions */
static PyObject* bind(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  PyObject** const to[6] = {&quantize_ctypes, &rmsnorm_quant_ctypes, &swiglu_quant_ctypes, &matmul_ctypes, &gemv_gu_ctypes, &layer_moe_ctypes};
  (void)self;
  if (nargs != 6) {
    PyErr_SetString(PyExc_TypeError, "bind takes the six functions");
    return NULL;
  }
  for (int i = 0; i < 6; ++i) {
    Py_INCREF(args[i]);
    Py_XSETREF(*to[i], args[i]);
  }
  Py_RETURN_NONE;
}

#define METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))NAME, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {METHOD(quantize), METHOD(rmsnorm_quant), METHOD(swiglu_quant), METHOD(matmul),
                                METHOD(gemv_gu), METHOD(layer_moe), METHOD(bind), {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pycall", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__pycall(void) { return PyModule_Create(&module); }
