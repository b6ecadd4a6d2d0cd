/*
 * _slmt_fast: a CPython METH_FASTCALL binding of the hot entry points of
 * libslmturbo_hip.so.  ctypes spends ~3 us converting a dozen arguments per call;
 * this module takes the same arguments as plain Python ints (pointers as integers)
 * and calls the library through function pointers that kernels/_native.py hands it
 * from the loaded library (bind), so the two bindings always reach the same code.
 * Host code only: no device work happens here.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/slmturbo.h"

/* args[i] as a 64-bit integer; -1 with an exception set on failure */
static int take(PyObject* const* args, Py_ssize_t n, long long* v) {
  for (Py_ssize_t i = 0; i < n; ++i) {
    v[i] = PyLong_AsLongLong(args[i]);
    if (v[i] == -1 && PyErr_Occurred()) return -1;
  }
  return 0;
}

#define P(i) ((void*)(intptr_t)v[i])
#define I(i) ((int)v[i])
#define L(i) ((int64_t)v[i])

/*
 * One function: N integer arguments, handed on as the entry point's own types.  Other
 * Python threads run meanwhile, as during a ctypes call (a first launch loads code, and
 * one on a full queue waits), where RUN is FREE.  The decodes keep the lock (HELD): they
 * share the stream's workspace, which the batched one fills in one launch and reads in
 * the next, and another thread's decode must not come between these.
 */
#define HELD(...) __VA_ARGS__
#define FREE(...) Py_BEGIN_ALLOW_THREADS __VA_ARGS__ Py_END_ALLOW_THREADS
#define ENTRY(name, RUN, N, ...)                                                   \
  static __typeof__(slmt_##name)* g_##name = NULL;                                 \
  static PyObject* name(PyObject* self, PyObject* const* args, Py_ssize_t n) {     \
    (void)self;                                                                    \
    long long v[N];                                                                \
    if (!g_##name) {                                                               \
      PyErr_SetString(PyExc_RuntimeError, #name ": library not bound");            \
      return NULL;                                                                 \
    }                                                                              \
    if (n != N) {                                                                  \
      PyErr_SetString(PyExc_TypeError, #name " takes " #N " arguments");           \
      return NULL;                                                                 \
    }                                                                              \
    if (take(args, N, v)) return NULL;                                             \
    long long rc;                                                                  \
    RUN(rc = g_##name(__VA_ARGS__);)                                               \
    return PyLong_FromLongLong(rc);                                                \
  }

ENTRY(quantize_store, HELD, 12, P(0), L(1), P(2), L(3), P(4), L(5), I(6), P(7), L(8), I(9), I(10), P(11))
ENTRY(decode_paged_batched, HELD, 22, P(0), L(1), L(2), P(3), L(4), I(5), P(6), I(7), L(8), P(9), I(10), I(11),
      I(12), I(13), I(14), P(15), I(16), L(17), L(18), P(19), L(20), P(21))
ENTRY(chunk_paged, FREE, 24, P(0), L(1), L(2), P(3), L(4), I(5), P(6), I(7), L(8), P(9), P(10), I(11), I(12), I(13),
      I(14), I(15), I(16), P(17), I(18), L(19), L(20), P(21), L(22), P(23))
ENTRY(chunk_workspace_bytes, HELD, 6, L(0), I(1), I(2), I(3), I(4), I(5))
ENTRY(decode_per_token, HELD, 17, P(0), P(1), P(2), P(3), P(4), P(5), P(6), I(7), I(8), I(9), I(10), I(11), I(12),
      P(13), P(14), L(15), P(16))
ENTRY(decode_per_channel, HELD, 18, P(0), P(1), P(2), P(3), P(4), P(5), P(6), I(7), I(8), I(9), I(10), I(11), I(12),
      I(13), P(14), P(15), L(16), P(17))
ENTRY(prefill_per_channel, FREE, 21, P(0), P(1), P(2), P(3), P(4), P(5), P(6), I(7), I(8), I(9), I(10), I(11),
      I(12), I(13), I(14), I(15), I(16), P(17), P(18), L(19), P(20))
ENTRY(quantize_kv_per_channel, FREE, 12, P(0), P(1), I(2), I(3), I(4), P(5), P(6), P(7), P(8), P(9), P(10), P(11))
ENTRY(quantize_with_rulers, FREE, 12, P(0), L(1), L(2), I(3), I(4), I(5), P(6), P(7), P(8), L(9), L(10), P(11))

/* bind(name, address): the library's entry point slmt_<name> */
static PyObject* bind(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  (void)self;
  long long at;
  if (n != 2 || !PyUnicode_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "bind(name, address)");
    return NULL;
  }
  if (take(args + 1, 1, &at)) return NULL;
  if (!at) {
    PyErr_SetString(PyExc_ValueError, "bind: null function address");
    return NULL;
  }
#define BIND(name)                                                  \
  if (PyUnicode_CompareWithASCIIString(args[0], #name) == 0) {      \
    g_##name = (__typeof__(slmt_##name)*)(intptr_t)at;              \
    Py_RETURN_NONE;                                                 \
  }
  BIND(quantize_store)
  BIND(decode_paged_batched)
  BIND(chunk_paged)
  BIND(chunk_workspace_bytes)
  BIND(decode_per_token)
  BIND(decode_per_channel)
  BIND(prefill_per_channel)
  BIND(quantize_kv_per_channel)
  BIND(quantize_with_rulers)
  PyErr_SetString(PyExc_ValueError, "bind: no such entry point");
  return NULL;
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, "slmt_" #name}
static PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, "bind one of the library's entry points"},
    METHOD(quantize_store),
    METHOD(decode_paged_batched),
    METHOD(chunk_paged),
    METHOD(chunk_workspace_bytes),
    METHOD(decode_per_token),
    METHOD(decode_per_channel),
    METHOD(prefill_per_channel),
    METHOD(quantize_kv_per_channel),
    METHOD(quantize_with_rulers),
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_slmt_fast", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__slmt_fast(void) { return PyModule_Create(&module); }
