/* Calls from Python into the library's launch entry points, without ctypes: an eager call of
 * a few-microsecond kernel is bound by its host path, and converting the ~27 arguments of a
 * launch took ctypes 2.4 us, this 0.5 us. Same functions, same arguments, same status; the
 * binding passes the addresses it looked up (bind), so there is one copy of the library.
 *
 * Integers convert as ctypes converts them (a Python int, or None for a null pointer, cut to
 * the parameter's width); the interpreter lock is released for the call.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <string.h>

#include "../../include/tinyserve_amd.h"

static int64_t as_int(PyObject* o) {
  return o == Py_None ? 0 : (int64_t)PyLong_AsUnsignedLongLongMask(o);
}

#define P(i) (void*)(uintptr_t)v[i].n
#define I(i) (int)v[i].n
#define L(i) v[i].n
#define F(i) v[i].f

typedef union {
  int64_t n;
  double f;
} Arg;

enum { kMaxArgs = 40 };

/* `kinds`: the argument list's macro names, whose letters say which are floating. */
static int convert(const char* name, const char* kinds, int want, PyObject* const* a, Py_ssize_t n, Arg* v) {
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "%s takes %d arguments, got %zd", name, want, n);
    return -1;
  }
  const char* k = kinds;
  for (int i = 0; i < want; ++i) {
    while (*k != 'P' && *k != 'I' && *k != 'L' && *k != 'F') ++k;
    if (*k++ == 'F') v[i].f = PyFloat_AsDouble(a[i]);
    else v[i].n = as_int(a[i]);
  }
  return PyErr_Occurred() ? -1 : 0;
}

#define ENTRY(NAME, N, ...)                                                          \
  static __typeof__(&NAME) p_##NAME;                                                 \
  static PyObject* call_##NAME(PyObject* self, PyObject* const* a, Py_ssize_t n) {   \
    Arg v[kMaxArgs];                                                                 \
    int rc;                                                                          \
    (void)self;                                                                      \
    if (!p_##NAME) {                                                                 \
      PyErr_SetString(PyExc_RuntimeError, #NAME " is not bound");                    \
      return NULL;                                                                   \
    }                                                                                \
    if (convert(#NAME, #__VA_ARGS__, N, a, n, v)) return NULL;                       \
    Py_BEGIN_ALLOW_THREADS                                                           \
    rc = p_##NAME(__VA_ARGS__);                                                      \
    Py_END_ALLOW_THREADS                                                             \
    return PyLong_FromLong(rc);                                                      \
  }

ENTRY(ts_decode_split, 27,
      P(0), P(1), P(2), P(3), P(4), P(5), P(6), P(7), P(8), I(9), I(10), I(11), I(12), I(13),
      L(14), L(15), L(16), L(17), L(18), L(19), L(20), I(21), I(22), I(23), F(24), I(25), P(26))
ENTRY(ts_decode_combine, 12,
      P(0), P(1), P(2), P(3), I(4), I(5), I(6), L(7), L(8), I(9), I(10), P(11))
ENTRY(ts_prefill_varlen_ws, 28,
      P(0), P(1), P(2), P(3), P(4), P(5), P(6), P(7), I(8), I(9), I(10), I(11), I(12), I(13),
      L(14), L(15), L(16), L(17), L(18), L(19), L(20), L(21), F(22), I(23), L(24), P(25), L(26),
      P(27))
ENTRY(ts_rms_norm_rows, 10,
      P(0), P(1), P(2), I(3), I(4), L(5), L(6), F(7), I(8), P(9))
ENTRY(ts_add_rms_norm_rows, 12,
      P(0), P(1), P(2), P(3), I(4), I(5), L(6), L(7), L(8), F(9), I(10), P(11))
ENTRY(ts_silu_mul, 8,
      P(0), P(1), I(2), I(3), L(4), L(5), I(6), P(7))
ENTRY(ts_qk_norm_rope_store, 30,
      P(0), P(1), P(2), P(3), P(4), P(5), P(6), P(7), P(8), P(9), P(10), I(11), I(12), I(13),
      I(14), L(15), L(16), L(17), L(18), L(19), L(20), L(21), L(22), L(23), L(24), L(25), F(26),
      I(27), I(28), P(29))
ENTRY(ts_rope_cos_sin, 8,
      P(0), I(1), I(2), F(3), P(4), P(5), L(6), P(7))
ENTRY(ts_rows_gemm, 15,
      P(0), I(1), L(2), P(3), L(4), P(5), L(6), P(7), L(8), I(9), I(10), I(11), I(12), I(13),
      P(14))
ENTRY(ts_add_rms_norm, 15,
      P(0), L(1), P(2), I(3), P(4), P(5), L(6), P(7), I(8), L(9), I(10), I(11), F(12), I(13),
      P(14))

#define EACH(X)                                                                     \
  X(ts_decode_split)                                                                \
  X(ts_decode_combine)                                                              \
  X(ts_prefill_varlen_ws)                                                           \
  X(ts_rms_norm_rows)                                                               \
  X(ts_add_rms_norm_rows)                                                           \
  X(ts_silu_mul)                                                                    \
  X(ts_qk_norm_rope_store)                                                          \
  X(ts_rope_cos_sin)                                                                \
  X(ts_rows_gemm)                                                                   \
  X(ts_add_rms_norm)

/* bind(name, address): where the library has the entry point. False for a name not here. */
static PyObject* bind(PyObject* self, PyObject* args) {
  const char* name;
  unsigned long long at;
  (void)self;
  if (!PyArg_ParseTuple(args, "sK", &name, &at)) return NULL;
#define BIND(NAME)                                          \
  if (strcmp(name, #NAME) == 0) {                           \
    p_##NAME = (__typeof__(&NAME))(uintptr_t)at;            \
    Py_RETURN_TRUE;                                         \
  }
  EACH(BIND)
  Py_RETURN_FALSE;
}

#define METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))call_##NAME, METH_FASTCALL, NULL},
static PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, NULL}, EACH(METHOD){NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__fastcall(void) { return PyModule_Create(&module); }
