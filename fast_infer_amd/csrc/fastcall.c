// Native call path of the Python wrappers: the library's hot entry points as CPython functions.
//
// A ctypes call converts every argument through a Python-level type object, 1.5 us for the 15
// arguments of fi_int4_matmul and 3.5 us for the 38 of fi_rope_store_kv, of the 7 to 10 us a wrapper
// takes; decode calls of few rows are bound by that time.  Here each argument is one integer
// conversion (about 0.2 and 0.4 us a call).  The functions are those of the library that
// _lib.load() opened: their addresses are bound after loading, nothing is linked here.  The
// interpreter lock is released during the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "../../include/fast_infer_amd.h"

// One argument list by its format: 'p' pointer (an integer address or None), 'i' integer, 'f'
// float.  Integers go to v in order, the float to *f.  0, or -1 with an exception set.
static int parse(const char* name, const char* fmt, PyObject* const* args, Py_ssize_t n, int64_t* v,
                 float* f) {
  if ((size_t)n != strlen(fmt)) {
    PyErr_Format(PyExc_TypeError, "%s takes %zu arguments, %zd given", name, strlen(fmt), n);
    return -1;
  }
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* a = args[i];
    if (fmt[i] == 'f') {
      const double d = PyFloat_AsDouble(a);
      if (d == -1.0 && PyErr_Occurred()) return -1;
      *f = (float)d;
    } else if (fmt[i] == 'p' && a == Py_None) {
      *v++ = 0;
    } else {
      const long long x = PyLong_AsLongLong(a);  // TypeError for anything without __index__
      if (x == -1 && PyErr_Occurred()) return -1;
      *v++ = x;
    }
  }
  return 0;
}

#define MAX_ARGS 40
#define CALL(name, fmt, ...)                                                            \
  static __typeof__(&name) name##_fn;                                                   \
  static PyObject* py_##name(PyObject* self, PyObject* const* args, Py_ssize_t n) {     \
    (void)self;                                                                         \
    _Static_assert(sizeof(fmt) <= MAX_ARGS + 1, "argument buffer");                      \
    int64_t v[MAX_ARGS];                                                                \
    float f = 0.f;                                                                      \
    int rc;                                                                             \
    if (!name##_fn) {                                                                   \
      PyErr_SetString(PyExc_RuntimeError, #name " is not bound");                       \
      return NULL;                                                                      \
    }                                                                                   \
    if (parse(#name, fmt, args, n, v, &f)) return NULL;                                 \
    (void)f;                                                                            \
    Py_BEGIN_ALLOW_THREADS rc = name##_fn(__VA_ARGS__);                                 \
    Py_END_ALLOW_THREADS return PyLong_FromLong(rc);                                    \
  }

CALL(fi_flash_attention_fwd, "ppppiiiiiiiiiiiiiiiiifppiipiip",
       (const void*)v[0], (const void*)v[1], (const void*)v[2], (void*)v[3], v[4], v[5],
       v[6], v[7], v[8], v[9], v[10], v[11], v[12], v[13], v[14], v[15], v[16], v[17],
       v[18], v[19], v[20], f, (void*)v[21], (void*)v[22], v[23], v[24], (const
       int32_t*)v[25], v[26], v[27], (void*)v[28])

CALL(fi_paged_attention_fwd, "piippiiipiipipiiiiifpip",
       (const void*)v[0], v[1], v[2], (const void*)v[3], (const void*)v[4], v[5], v[6],
       v[7], (const int32_t*)v[8], v[9], v[10], (const int32_t*)v[11], v[12], (void*)v[13],
       v[14], v[15], v[16], v[17], v[18], f, (void*)v[19], (size_t)v[20], (void*)v[21])

CALL(fi_rope_store_kv, "piiipiiipiiippipiiipiiippiipiiiiiiiipp",
       (const void*)v[0], v[1], v[2], v[3], (const void*)v[4], v[5], v[6], v[7], (const
       void*)v[8], v[9], v[10], v[11], (const void*)v[12], (const void*)v[13], v[14],
       (void*)v[15], v[16], v[17], v[18], (void*)v[19], v[20], v[21], v[22], (void*)v[23],
       (void*)v[24], v[25], v[26], (const int32_t*)v[27], v[28], v[29], v[30], v[31], v[32],
       v[33], v[34], v[35], (const int32_t*)v[36], (void*)v[37])

CALL(fi_int4_matmul, "piiipipiiipipip",
       (const void*)v[0], v[1], v[2], v[3], (const void*)v[4], v[5], (const void*)v[6],
       v[7], v[8], v[9], (void*)v[10], v[11], (void*)v[12], (size_t)v[13], (void*)v[14])

CALL(fi_rmsnorm, "piiipfpip",
       (const void*)v[0], v[1], v[2], v[3], (const void*)v[4], f, (void*)v[5], v[6],
       (void*)v[7])

CALL(fi_rmsnorm_int4_matmul, "piiipfpipiiipipip",
       (const void*)v[0], v[1], v[2], v[3], (const void*)v[4], f, (const void*)v[5], v[6],
       (const void*)v[7], v[8], v[9], v[10], (void*)v[11], v[12], (void*)v[13],
       (size_t)v[14], (void*)v[15])

#define NAMES(X)           \
  X(fi_flash_attention_fwd) \
  X(fi_paged_attention_fwd) \
  X(fi_rope_store_kv) \
  X(fi_int4_matmul) \
  X(fi_rmsnorm) \
  X(fi_rmsnorm_int4_matmul)

// bind(name, address): the entry point `name` of the loaded library.
static PyObject* bind(PyObject* self, PyObject* args) {
  (void)self;
  const char* name;
  unsigned long long addr;
  if (!PyArg_ParseTuple(args, "sK", &name, &addr)) return NULL;
#define BIND(fn)                                   \
  if (!strcmp(name, #fn)) {                        \
    fn##_fn = (__typeof__(&fn))(uintptr_t)addr;    \
    Py_RETURN_NONE;                                \
  }
  NAMES(BIND)
  PyErr_Format(PyExc_ValueError, "no entry point %s", name);
  return NULL;
}

#define METHOD(fn) {#fn, (PyCFunction)(void (*)(void))py_##fn, METH_FASTCALL, NULL},
static PyMethodDef methods[] = {NAMES(METHOD) {"bind", bind, METH_VARARGS, NULL}, {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", NULL, -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__fastcall(void) { return PyModule_Create(&module); }
