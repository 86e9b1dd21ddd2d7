// Calls of the kernel libraries' entry points from Python without ctypes. A step that is not replayed from a graph makes some 250 of
// them with up to 40 arguments each; ctypes converts every argument through objects of its own and costs 2-3 us a call beside the
// launch's 2.3, which is what bounds such steps (489 prompt tokens beside 23 decoding requests at the 0.6B sizes).
//
//   bind(address, signature, fallback) -> callable   signature: a letter per argument, i an integer or pointer (None: null), f a float
//   caller(functions, failed) -> callable            caller(name, *args): functions[name](*args), and failed(name) if that is not 0
//
// Arguments go out as the x86-64 System V convention wants them whatever their order: integers and pointers in the six integer
// registers and then on the stack, up to eight floats in the vector registers, none on the stack. So one function type serves
// all entry points: what a callee does not take is ignored, the caller clears the stack, and a callee that takes 32 bits reads the
// lower half. A call whose arguments are anything else (an array of ctypes, another number of them) goes to `fallback`, the ctypes function, which converts or
// refuses it as before. The interpreter is released for the time of a call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <cstddef>
#include <cstdint>
#include <cstring>

#if !defined(__x86_64__)
#error "the entry points are called by the x86-64 System V convention"
#endif

constexpr int MAX_INTS = 48, MAX_FLOATS = 8, MAX_ARGS = MAX_INTS + MAX_FLOATS;
#define I6 int64_t, int64_t, int64_t, int64_t, int64_t, int64_t
typedef int (*entry_t)(I6, I6, I6, I6, I6, I6, I6, I6, float, float, float, float, float, float, float, float);

struct Call {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  entry_t entry;
  PyObject* fallback;
  int count;
  char kinds[MAX_ARGS];
};

// The entry point's result, or -1 with an exception set in *raised.
static long run(Call* c, PyObject* const* args, bool* raised, PyObject** other, size_t nargs) {
  int64_t n[MAX_INTS] = {0};
  float f[MAX_FLOATS] = {0.f};
  int ints = 0, floats = 0;
  *raised = false;
  *other = nullptr;
  bool plain = (Py_ssize_t)nargs == c->count;
  for (int i = 0; plain && i < c->count; ++i) {
    PyObject* a = args[i];
    if (c->kinds[i] == 'f') {
      if (PyFloat_Check(a)) f[floats++] = (float)PyFloat_AS_DOUBLE(a);
      else plain = false;
    } else if (a == Py_None) {
      n[ints++] = 0;
      plain = c->kinds[i] == 'p';
    } else if (PyLong_Check(a)) {
      const unsigned long long v = PyLong_AsUnsignedLongLongMask(a);
      if (v == (unsigned long long)-1 && PyErr_Occurred()) { *raised = true; return -1; }
      n[ints++] = (int64_t)v;
    } else {
      plain = false;
    }
  }
  if (!plain) {
    *other = PyObject_Vectorcall(c->fallback, args, nargs, nullptr);
    *raised = *other == nullptr;
    return -1;
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = c->entry(n[0], n[1], n[2], n[3], n[4], n[5], n[6], n[7], n[8], n[9], n[10], n[11], n[12], n[13], n[14], n[15], n[16], n[17], n[18],
                n[19], n[20], n[21], n[22], n[23], n[24], n[25], n[26], n[27], n[28], n[29], n[30], n[31], n[32], n[33], n[34], n[35],
                n[36], n[37], n[38], n[39], n[40], n[41], n[42], n[43], n[44], n[45], n[46], n[47], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
  Py_END_ALLOW_THREADS
  return rc;
}

static PyObject* call_vector(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  if (kwnames && PyTuple_GET_SIZE(kwnames)) { PyErr_SetString(PyExc_TypeError, "entry points take no keywords"); return nullptr; }
  bool raised;
  PyObject* other;
  const long rc = run((Call*)self, args, &raised, &other, PyVectorcall_NARGS(nargsf));
  if (raised) return nullptr;
  return other ? other : PyLong_FromLong(rc);
}
static void call_dealloc(PyObject* self) {
  Py_XDECREF(((Call*)self)->fallback);
  Py_TYPE(self)->tp_free(self);
}
static PyTypeObject CallType = {PyVarObject_HEAD_INIT(nullptr, 0) "me_calls.Call", sizeof(Call)};

struct Caller {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  PyObject *functions, *failed;
};
static PyObject* caller_vector(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  Caller* c = (Caller*)self;
  const Py_ssize_t nargs = PyVectorcall_NARGS(nargsf);
  if (nargs < 1 || (kwnames && PyTuple_GET_SIZE(kwnames))) { PyErr_SetString(PyExc_TypeError, "call(name, *args)"); return nullptr; }
  PyObject* fn = PyDict_GetItemWithError(c->functions, args[0]);
  if (!fn) {
    if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, args[0]);
    return nullptr;
  }
  Py_INCREF(fn);
  bool raised = false, ok;
  PyObject* other = nullptr;
  long rc = -1;
  if (Py_TYPE(fn) == &CallType) {
    rc = run((Call*)fn, args + 1, &raised, &other, nargs - 1);
  } else {
    other = PyObject_Vectorcall(fn, args + 1, nargs - 1, nullptr);
    raised = other == nullptr;
  }
  Py_DECREF(fn);
  if (raised) return nullptr;
  if (other) {
    rc = PyLong_AsLong(other);
    Py_DECREF(other);
    if (rc == -1 && PyErr_Occurred()) return nullptr;
  }
  ok = rc == 0;
  if (ok) Py_RETURN_NONE;
  return PyObject_CallOneArg(c->failed, args[0]);
}
static void caller_dealloc(PyObject* self) {
  Py_XDECREF(((Caller*)self)->functions);
  Py_XDECREF(((Caller*)self)->failed);
  Py_TYPE(self)->tp_free(self);
}
static PyTypeObject CallerType = {PyVarObject_HEAD_INIT(nullptr, 0) "me_calls.Caller", sizeof(Caller)};

static PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long address;
  const char* kinds;
  Py_ssize_t count;
  PyObject* fallback;
  if (!PyArg_ParseTuple(args, "Ks#O", &address, &kinds, &count, &fallback)) return nullptr;
  int ints = 0, floats = 0;
  for (Py_ssize_t i = 0; i < count; ++i) {
    if (kinds[i] == 'f') ++floats;
    else if (kinds[i] == 'i' || kinds[i] == 'p') ++ints;
    else { PyErr_SetString(PyExc_ValueError, "a signature has i, p and f"); return nullptr; }
  }
  if (ints > MAX_INTS || floats > MAX_FLOATS) { Py_INCREF(fallback); return fallback; }
  Call* c = PyObject_New(Call, &CallType);
  if (!c) return nullptr;
  c->vectorcall = call_vector;
  c->entry = reinterpret_cast<entry_t>((uintptr_t)address);
  Py_INCREF(fallback);
  c->fallback = fallback;
  c->count = (int)count;
  memcpy(c->kinds, kinds, count);
  return (PyObject*)c;
}
static PyObject* caller(PyObject*, PyObject* args) {
  PyObject *functions, *failed;
  if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &functions, &failed)) return nullptr;
  Caller* c = PyObject_New(Caller, &CallerType);
  if (!c) return nullptr;
  c->vectorcall = caller_vector;
  Py_INCREF(functions); Py_INCREF(failed);
  c->functions = functions; c->failed = failed;
  return (PyObject*)c;
}

static PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr}, {"caller", caller, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
static PyModuleDef module = {PyModuleDef_HEAD_INIT, "me_calls", nullptr, -1, methods};

PyMODINIT_FUNC PyInit_me_calls() {
  CallType.tp_flags = CallerType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  CallType.tp_call = CallerType.tp_call = PyVectorcall_Call;
  CallType.tp_vectorcall_offset = offsetof(Call, vectorcall);
  CallerType.tp_vectorcall_offset = offsetof(Caller, vectorcall);
  CallType.tp_dealloc = call_dealloc;
  CallerType.tp_dealloc = caller_dealloc;
  if (PyType_Ready(&CallType) < 0 || PyType_Ready(&CallerType) < 0) return nullptr;
  return PyModule_Create(&module);
}
