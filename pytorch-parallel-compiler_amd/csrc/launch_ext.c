/* CPython extension _wc_launch: calls a C-ABI entry point of libwide_hip.so of the form
 *   int32_t entry(const args*, void* stream)
 * by address.  A ctypes call costs about 3 us on the host, most of a small wide forward's
 * dispatch time; this call costs a fraction of that.  The caller passes the entry point's
 * address, the address of its filled argument block and the stream handle as integers.  Like a
 * ctypes call, the entry points run without the interpreter lock (a launch can wait in the runtime
 * when its queue is full); call2 alone holds it, because its block belongs to the module and
 * another thread's forward may fill it next. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

typedef int32_t (*wc_entry2)(const void*, void*);

static PyObject* call2(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  (void)self;
  if (nargs != 3) {
    PyErr_SetString(PyExc_TypeError, "call2(entry, args, stream) takes 3 integer arguments");
    return NULL;
  }
  void* fn = PyLong_AsVoidPtr(args[0]);
  void* a = PyLong_AsVoidPtr(args[1]);
  void* s = PyLong_AsVoidPtr(args[2]);
  if (PyErr_Occurred()) return NULL;
  if (!fn || !a) {
    PyErr_SetString(PyExc_ValueError, "call2: null entry point or argument block");
    return NULL;
  }
  return PyLong_FromLong((long)((wc_entry2)fn)(a, s));
}

/* callb(entry, block, stream): the argument block as a bytes object (struct.pack of the C struct's
 * fields; the caller checks its size once), read in place. */
static PyObject* callb(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  (void)self;
  if (nargs != 3 || !PyBytes_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "callb(entry, block, stream) takes an integer, bytes and an integer");
    return NULL;
  }
  void* fn = PyLong_AsVoidPtr(args[0]);
  void* s = PyLong_AsVoidPtr(args[2]);
  if (PyErr_Occurred()) return NULL;
  if (!fn) {
    PyErr_SetString(PyExc_ValueError, "callb: null entry point");
    return NULL;
  }
  const void* block = PyBytes_AS_STRING(args[1]);      /* the caller's reference outlives the call */
  int32_t rc;
  Py_BEGIN_ALLOW_THREADS
  rc = ((wc_entry2)fn)(block, s);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong((long)rc);
}

typedef int32_t (*wc_layernorm_t)(const void*, int64_t, int64_t, const void*, const void*, void*, int64_t, int64_t,
                                  int64_t, int64_t, int64_t, float, int32_t, int32_t, void*);

/* layernorm(entry, x, x_model_stride, x_row_stride, gamma, beta, y, y_model_stride, y_row_stride, n,
 * rows_per_model, dim, eps, dtype, param_dtype, stream): wc_layernorm, whose arguments are passed
 * one by one. */
static PyObject* layernorm(PyObject* self, PyObject* const* a, Py_ssize_t nargs) {
  (void)self;
  if (nargs != 16) {
    PyErr_SetString(PyExc_TypeError, "layernorm takes 16 arguments");
    return NULL;
  }
  void* fn = PyLong_AsVoidPtr(a[0]);
  void *x = PyLong_AsVoidPtr(a[1]), *g = PyLong_AsVoidPtr(a[4]), *b = PyLong_AsVoidPtr(a[5]),
       *y = PyLong_AsVoidPtr(a[6]), *st = PyLong_AsVoidPtr(a[15]);
  int64_t i[7];
  static const int at[7] = {2, 3, 7, 8, 9, 10, 11};
  for (int k = 0; k < 7; ++k) i[k] = PyLong_AsLongLong(a[at[k]]);
  const double eps = PyFloat_AsDouble(a[12]);
  const long dt = PyLong_AsLong(a[13]), pdt = PyLong_AsLong(a[14]);
  if (PyErr_Occurred()) return NULL;
  if (!fn) {
    PyErr_SetString(PyExc_ValueError, "layernorm: null entry point");
    return NULL;
  }
  int32_t rc;
  Py_BEGIN_ALLOW_THREADS
  rc = ((wc_layernorm_t)fn)(x, i[0], i[1], g, b, y, i[2], i[3], i[4], i[5], i[6], (float)eps, (int32_t)dt,
                            (int32_t)pdt, st);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong((long)rc);
}

typedef int32_t (*wc_conv_pack_t)(const void*, int64_t, int64_t, int64_t, int64_t, int64_t, int32_t, void*, void*);

/* conv_pack(entry, w, n, c_out, c_in, kh, kw, dtype, out, stream): wc_conv_pack_weights */
static PyObject* conv_pack(PyObject* self, PyObject* const* a, Py_ssize_t nargs) {
  (void)self;
  if (nargs != 10) {
    PyErr_SetString(PyExc_TypeError, "conv_pack takes 10 arguments");
    return NULL;
  }
  void *fn = PyLong_AsVoidPtr(a[0]), *w = PyLong_AsVoidPtr(a[1]), *out = PyLong_AsVoidPtr(a[8]),
       *st = PyLong_AsVoidPtr(a[9]);
  int64_t i[5];
  for (int k = 0; k < 5; ++k) i[k] = PyLong_AsLongLong(a[2 + k]);
  const long dt = PyLong_AsLong(a[7]);
  if (PyErr_Occurred()) return NULL;
  if (!fn) {
    PyErr_SetString(PyExc_ValueError, "conv_pack: null entry point");
    return NULL;
  }
  int32_t rc;
  Py_BEGIN_ALLOW_THREADS
  rc = ((wc_conv_pack_t)fn)(w, i[0], i[1], i[2], i[3], i[4], (int32_t)dt, out, st);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong((long)rc);
}

static PyMethodDef methods[] = {
    {"call2", (PyCFunction)(void (*)(void))call2, METH_FASTCALL,
     "call2(entry, args, stream) -> status: entry(args, stream) for addresses given as integers"},
    {"callb", (PyCFunction)(void (*)(void))callb, METH_FASTCALL,
     "callb(entry, block, stream) -> status: entry(block's bytes, stream)"},
    {"layernorm", (PyCFunction)(void (*)(void))layernorm, METH_FASTCALL,
     "layernorm(entry, the 15 arguments of wc_layernorm) -> status"},
    {"conv_pack", (PyCFunction)(void (*)(void))conv_pack, METH_FASTCALL,
     "conv_pack(entry, the 9 arguments of wc_conv_pack_weights) -> status"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_wc_launch", NULL, -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__wc_launch(void) { return PyModule_Create(&module); }
