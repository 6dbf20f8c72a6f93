/* Calls from Python into the library's launch entry points, without ctypes: an eager call of
 * a few-microsecond kernel is bound by its host path, and converting the ~27 arguments of a
 * launch took ctypes 2.4 us, this 0.5 us. Same functions, same arguments, same status; the
 * binding passes the addresses it looked up (bind), so there is one copy of the library.
 *
 * Integers convert as ctypes converts them (a Python int, cut to the parameter's width; None
 * for a null pointer only), floats as PyFloat_AsDouble takes them; the interpreter lock is
 * released for the call.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <string.h>

#include "../../include/tinyserve_amd.h"

#define P(i) (void*)(uintptr_t)v[i].n
#define I(i) (int)v[i].n
#define L(i) v[i].n
#define F(i) v[i].f

typedef union {
  int64_t n;
  double f;
} Arg;

enum { kMaxArgs = 40 };

/* The next argument's kind (P, I, L or F; 0 at the end) of a list of macro names. */
static char next_kind(const char** kinds) {
  for (; **kinds; ++*kinds)
    if (strchr("PILF", **kinds)) return *(*kinds)++;
  return 0;
}

/* `kinds`: each argument's. */
static int convert(const char* name, const char* kinds, int want, PyObject* const* a, Py_ssize_t n, Arg* v) {
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "%s takes %d arguments, got %zd", name, want, n);
    return -1;
  }
  for (int i = 0; i < want; ++i) {
    const char k = kinds[i];
    if (k == 'F') {
      v[i].f = PyFloat_AsDouble(a[i]);
      if (v[i].f == -1.0 && PyErr_Occurred()) return -1;
    } else if (k == 'P' && a[i] == Py_None) {
      v[i].n = 0;
    } else {
      v[i].n = (int64_t)PyLong_AsUnsignedLongLongMask(a[i]);
      if (v[i].n == -1 && PyErr_Occurred()) return -1;
    }
  }
  return 0;
}

#define ENTRY(NAME, N, ...)                                                          \
  static __typeof__(&NAME) p_##NAME;                                                 \
  static const char list_##NAME[] = #__VA_ARGS__;                                    \
  static char k_##NAME[kMaxArgs]; /* its kinds, from bind */                         \
  static PyObject* call_##NAME(PyObject* self, PyObject* const* a, Py_ssize_t n) {   \
    Arg v[kMaxArgs];                                                                 \
    int rc;                                                                          \
    (void)self;                                                                      \
    if (!p_##NAME) {                                                                 \
      PyErr_SetString(PyExc_RuntimeError, #NAME " is not bound");                    \
      return NULL;                                                                   \
    }                                                                                \
    if (convert(#NAME, k_##NAME, N, a, n, v)) return NULL;                           \
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

/* Whether an argument list's letters are `want`, letter for letter. */
static int same_kinds(const char* kinds, const char* want) {
  char k;
  while ((k = next_kind(&kinds)) && k == *want) ++want;
  return k == 0 && *want == 0;
}

/* bind(name, address, kinds): where the library has the entry point, and the kinds of its
 * arguments ("PPIL..."). False, unbound, for a name that is not here or has others. */
static PyObject* bind(PyObject* self, PyObject* args) {
  const char *name, *kinds;
  unsigned long long at;
  (void)self;
  if (!PyArg_ParseTuple(args, "sKs", &name, &at, &kinds)) return NULL;
#define BIND(NAME)                                          \
  if (strcmp(name, #NAME) == 0) {                           \
    if (!same_kinds(list_##NAME, kinds)) Py_RETURN_FALSE;   \
    strcpy(k_##NAME, kinds);                                \
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
