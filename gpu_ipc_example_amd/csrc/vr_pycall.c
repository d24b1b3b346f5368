/* The three collective calls for Python: pointer lists into stack tables, one C ABI call.
 *
 * A collective call at launch-bound sizes costs what the host spends on it.  Through
 * ctypes that was 5.5 us a call, over half of it spent on turning lists into c_void_p
 * arrays and arguments into C types; the call itself is one kernel launch (2.3 us).
 * Everything else of the C ABI stays with ctypes (binding.py), which also holds the
 * argument checks, the context and the error texts: these functions return the status. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "vrank_allreduce.h"

/* Device addresses of a sequence; unused entries stay null.  -1 with an exception set.
 * Turning anything but an int into an address runs the caller's code, which may change the
 * caller's sequence: those are read from a tuple that is nobody else's. */
static int fill_table(PyObject *seq, void *table[VR_MAX_RANKS]) {
  for (int i = 0; i < VR_MAX_RANKS; ++i) table[i] = NULL;
  if (PyList_CheckExact(seq) || PyTuple_CheckExact(seq)) {
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
    PyObject *const *items = PySequence_Fast_ITEMS(seq);
    Py_ssize_t i = 0;
    for (; i < n && PyLong_CheckExact(items[i]); ++i)
      if (i < VR_MAX_RANKS)   /* no context looks further */
        table[i] = (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(items[i]);
    if (i == n) return 0;
  }
  PyObject *own = PySequence_Tuple(seq);
  if (!own) return -1;
  const Py_ssize_t n = PyTuple_GET_SIZE(own);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject *number = PyNumber_Long(PyTuple_GET_ITEM(own, i));
    if (!number) break;
    if (i < VR_MAX_RANKS) table[i] = (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(number);
    Py_DECREF(number);
  }
  Py_DECREF(own);
  return PyErr_Occurred() ? -1 : 0;
}

/* Of the module ctypes: what converts an argument that is not a plain int. */
static PyObject *ct_cast, *ct_void_p, *ct_size_t, *ct_int, *ct_error;

/* A hipStream_t as ctypes takes a c_void_p argument.  None (the null stream), an int and a
 * c_void_p are read here; ctypes converts the rest (objects with an _as_parameter_, pointers,
 * ...) or refuses it.  -1 with an exception set. */
static int stream_of(PyObject *o, void **stream) {
  *stream = NULL;
  if (o == Py_None) return 0;
  PyObject *pointer = NULL, *value = NULL;
  if (!PyLong_CheckExact(o)) {
    if (Py_TYPE(o) != (PyTypeObject *)ct_void_p) {
      pointer = PyObject_CallFunctionObjArgs(ct_cast, o, ct_void_p, NULL);
      if (!pointer) return -1;
      o = pointer;
    }
    o = value = PyObject_GetAttrString(o, "value");
  }
  if (o && o != Py_None) *stream = (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(o);
  Py_XDECREF(value);
  Py_XDECREF(pointer);
  return PyErr_Occurred() ? -1 : 0;
}

/* A number as ctypes takes an argument of the integer type `type`: an int (or what has an
 * __index__), a `type`, or an object that has one of these as its _as_parameter_.  -1 with an
 * exception set. */
static int number_of(PyObject *o, PyObject *type, unsigned long long *number) {
  if (PyLong_Check(o) || PyIndex_Check(o)) {
    *number = PyLong_AsUnsignedLongLongMask(o);
    return PyErr_Occurred() ? -1 : 0;
  }
  const int holds = PyObject_IsInstance(o, type);
  PyObject *inner = holds < 0 ? NULL : PyObject_GetAttrString(o, holds ? "value" : "_as_parameter_");
  if (!inner) {
    if (holds == 0 && PyErr_ExceptionMatches(PyExc_AttributeError))
      PyErr_Format(ct_error, "a number cannot be made of a %s", Py_TYPE(o)->tp_name);
    return -1;
  }
  int rc = Py_EnterRecursiveCall(" while converting an argument") ? -1 : 0;
  if (!rc) {
    rc = number_of(inner, type, number);
    Py_LeaveRecursiveCall();
  }
  Py_DECREF(inner);
  return rc;
}

/* The status of looking the name up; -1 with an exception set. */
static int algo_of(PyObject *name, int *algo) {
  const char *text = PyUnicode_AsUTF8(name);
  return text ? vr_algo_from_string(text, algo) : -1;
}

/* (context, sequence number, algo name, transport, inputs, outputs or None, nelems, stream) -> status.
 * The context is an address, the sequence number a writable buffer of 4 bytes (a ctypes c_uint32). */
static PyObject *collective(PyObject *const *args, Py_ssize_t nargs, int gather) {
  if (nargs != 8) {
    PyErr_SetString(PyExc_TypeError, "8 arguments expected");
    return NULL;
  }
  void *ins[VR_MAX_RANKS], *outs[VR_MAX_RANKS], *stream;
  int algo = -1, rc = algo_of(args[2], &algo);
  if (rc) return rc < 0 ? NULL : PyLong_FromLong(rc);
  vr_ctx *ctx = (vr_ctx *)(uintptr_t)PyLong_AsUnsignedLongLongMask(args[0]);
  unsigned long long transport, nelems;
  if (PyErr_Occurred() || number_of(args[3], ct_int, &transport) || number_of(args[6], ct_size_t, &nelems) ||
      stream_of(args[7], &stream))
    return NULL;
  const int in_place = args[5] == Py_None;
  if (fill_table(args[4], ins) || (!in_place && fill_table(args[5], outs))) return NULL;
  Py_buffer seq;
  if (PyObject_GetBuffer(args[1], &seq, PyBUF_WRITABLE)) return NULL;
  if (seq.len != (Py_ssize_t)sizeof(uint32_t)) {
    PyBuffer_Release(&seq);
    PyErr_SetString(PyExc_ValueError, "the sequence number has 4 bytes");
    return NULL;
  }
  Py_BEGIN_ALLOW_THREADS
  if (gather)
    rc = vr_allgather(ctx, stream, algo, (int)transport, (const void *const *)ins, in_place ? NULL : outs, (size_t)nelems,
                      (uint32_t *)seq.buf);
  else
    rc = vr_allreduce(ctx, stream, algo, (int)transport, ins, in_place ? NULL : outs, (size_t)nelems,
                      (uint32_t *)seq.buf);
  Py_END_ALLOW_THREADS
  PyBuffer_Release(&seq);
  return PyLong_FromLong(rc);
}

static PyObject *allreduce(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
  (void)self;
  return collective(args, nargs, 0);
}

static PyObject *allgather(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
  (void)self;
  return collective(args, nargs, 1);
}

/* (context, algo name, inputs, outputs or None, nelems, stream) -> status */
static PyObject *allreduce_static(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
  (void)self;
  if (nargs != 6) {
    PyErr_SetString(PyExc_TypeError, "6 arguments expected");
    return NULL;
  }
  void *ins[VR_MAX_RANKS], *outs[VR_MAX_RANKS], *stream;
  int algo = -1, rc = algo_of(args[1], &algo);
  if (rc) return rc < 0 ? NULL : PyLong_FromLong(rc);
  vr_ctx *ctx = (vr_ctx *)(uintptr_t)PyLong_AsUnsignedLongLongMask(args[0]);
  unsigned long long nelems;
  if (PyErr_Occurred() || number_of(args[4], ct_size_t, &nelems) || stream_of(args[5], &stream)) return NULL;
  const int in_place = args[3] == Py_None;
  if (fill_table(args[2], ins) || (!in_place && fill_table(args[3], outs))) return NULL;
  Py_BEGIN_ALLOW_THREADS
  rc = vr_allreduce_static(ctx, stream, algo, ins, in_place ? NULL : outs, (size_t)nelems);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

static PyMethodDef methods[] = {
    {"allreduce", (PyCFunction)(void (*)(void))allreduce, METH_FASTCALL, "vr_allreduce"},
    {"allgather", (PyCFunction)(void (*)(void))allgather, METH_FASTCALL, "vr_allgather"},
    {"allreduce_static", (PyCFunction)(void (*)(void))allreduce_static, METH_FASTCALL, "vr_allreduce_static"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", "Collective calls of the C ABI.", -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__call(void) {
  PyObject *ct = PyImport_ImportModule("ctypes");
  if (!ct) return NULL;
  ct_cast = PyObject_GetAttrString(ct, "cast");
  ct_void_p = PyObject_GetAttrString(ct, "c_void_p");
  ct_size_t = PyObject_GetAttrString(ct, "c_size_t");
  ct_int = PyObject_GetAttrString(ct, "c_int");
  ct_error = PyObject_GetAttrString(ct, "ArgumentError");
  Py_DECREF(ct);
  return ct_cast && ct_void_p && ct_size_t && ct_int && ct_error ? PyModule_Create(&module) : NULL;
}
