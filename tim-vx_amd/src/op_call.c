/* tvx_call: the Python binding's one hot call, tvx_op_run, without ctypes. On small layers a pass waits for the host's launches, and
 * a closure, a function call and five conversions stood in front of each: a pass of one launch 3.9 -> 3.3 us, of two 7.3 -> 6.5. The
 * function comes in by address: this module links against nothing. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

typedef int (*RunFn)(void*, const void*, const void*, void*, void*);

static RunFn run_fn;
static PyObject *data_ptr_name, *value_name, *pointer_type;

/* An address from None, a whole number or a c_void_p: 1; 0 for anything else, which is for ctypes to take or refuse; -1: an error. */
static int Address(PyObject* o, void** p) {
  *p = NULL;
  if (o == Py_None) return 1;
  if (PyLong_Check(o)) {
    *p = (void*)PyLong_AsUnsignedLongLongMask(o);
    return 1;
  }
  if ((PyObject*)Py_TYPE(o) != pointer_type) return 0;
  PyObject* v = PyObject_GetAttr(o, value_name);
  if (!v) return -1;
  if (v != Py_None) *p = (void*)PyLong_AsUnsignedLongLongMask(v);
  Py_DECREF(v);
  return 1;
}

/* ... or from a tensor's data_ptr() */
static int TensorAddress(PyObject* o, void** p) {
  if (o == Py_None || PyLong_Check(o)) return Address(o, p);
  PyObject* v = PyObject_CallMethodNoArgs(o, data_ptr_name);
  if (!v) return -1;
  const int ok = Address(v, p);
  Py_DECREF(v);
  return ok;
}

/* run(handle, in0, in1, out, stream) -> status, or NotImplemented for what only ctypes knows */
static PyObject* Run(PyObject* self, PyObject* const* args, Py_ssize_t count) {
  void* p[5];
  if (count != 5 || !run_fn) {
    PyErr_SetString(PyExc_TypeError, "run(handle, in0, in1, out, stream), after bind()");
    return NULL;
  }
  int known = 1;
  for (int i = 1; i < 6; ++i) {
    const int at = i % 5, ok = at % 4 ? TensorAddress(args[at], &p[at]) : Address(args[at], &p[at]);
    if (ok < 0) return NULL;
    known &= ok;
  }
  if (!known) Py_RETURN_NOTIMPLEMENTED;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = run_fn(p[0], p[1], p[2], p[3], p[4]);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

/* bind(address of tvx_op_run, ctypes.c_void_p) */
static PyObject* Bind(PyObject* self, PyObject* args) {
  PyObject *address, *type;
  if (!PyArg_ParseTuple(args, "OO", &address, &type)) return NULL;
  void* p = PyLong_AsVoidPtr(address);
  if (!p && PyErr_Occurred()) return NULL;
  Py_INCREF(type);
  Py_XSETREF(pointer_type, type);
  run_fn = (RunFn)p;
  Py_RETURN_NONE;
}

static PyMethodDef methods[] = {
    {"run", (PyCFunction)(void (*)(void))Run, METH_FASTCALL, "run(handle, in0, in1, out, stream) -> status"},
    {"bind", Bind, METH_VARARGS, "bind(address of tvx_op_run, ctypes.c_void_p)"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "tvx_call", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit_tvx_call(void) {
  data_ptr_name = PyUnicode_InternFromString("data_ptr");
  value_name = PyUnicode_InternFromString("value");
  return data_ptr_name && value_name ? PyModule_Create(&module) : NULL;
}
