/* tvx_call: the Python binding's one hot call, tvx_op_run, without ctypes. On small layers a pass waits for the host's launches, and
 * a closure, a function call and five conversions stood in front of each: a pass of one launch 3.9 -> 3.3 us, of two 7.3 -> 6.5. The
 * function comes in by address: this module links against nothing. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

typedef int (*RunFn)(void*, const void*, const void*, void*, void*);

static RunFn run_fn;
static PyObject *data_ptr_name, *value_name;

/* An address from None, a whole number, or attribute data_ptr() of a tensor / value of a ctypes pointer. */
static int Address(PyObject* o, int tensor, void** p) {
  *p = NULL;
  if (o == Py_None) return 1;
  if (PyLong_Check(o)) {
    *p = (void*)PyLong_AsUnsignedLongLongMask(o);
    return 1;
  }
  PyObject* v = tensor ? PyObject_CallMethodNoArgs(o, data_ptr_name) : PyObject_GetAttr(o, value_name);
  if (!v) return 0;
  const int ok = v == Py_None || PyLong_Check(v);
  if (ok && v != Py_None) *p = (void*)PyLong_AsUnsignedLongLongMask(v);
  Py_DECREF(v);
  if (!ok) PyErr_SetString(PyExc_TypeError, "no address");
  return ok;
}

/* run(handle, in0, in1, out, stream) -> status, or NotImplemented for a handle or stream of another type */
static PyObject* Run(PyObject* self, PyObject* const* args, Py_ssize_t count) {
  void* p[5];
  if (count != 5 || !run_fn) {
    PyErr_SetString(PyExc_TypeError, "run(handle, in0, in1, out, stream), after bind()");
    return NULL;
  }
  for (int i = 1; i < 4; ++i)
    if (!Address(args[i], 1, &p[i])) return NULL;
  for (int i = 0; i < 5; i += 4)
    if (!Address(args[i], 0, &p[i])) {  /* (whatever else ctypes takes for a pointer) */
      PyErr_Clear();
      Py_RETURN_NOTIMPLEMENTED;
    }
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = run_fn(p[0], p[1], p[2], p[3], p[4]);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

/* bind(address of tvx_op_run) */
static PyObject* Bind(PyObject* self, PyObject* address) {
  void* p = PyLong_AsVoidPtr(address);
  if (!p && PyErr_Occurred()) return NULL;
  run_fn = (RunFn)p;
  Py_RETURN_NONE;
}

static PyMethodDef methods[] = {
    {"run", (PyCFunction)(void (*)(void))Run, METH_FASTCALL, "run(handle, in0, in1, out, stream) -> status"},
    {"bind", Bind, METH_O, "bind(address of tvx_op_run)"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "tvx_call", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit_tvx_call(void) {
  data_ptr_name = PyUnicode_InternFromString("data_ptr");
  value_name = PyUnicode_InternFromString("value");
  return data_ptr_name && value_name ? PyModule_Create(&module) : NULL;
}
