/* Calls of the C ABI from Python without the conversions of ctypes, which take longer than the library needs to queue a short
 * call (1.0 us a call against 0.27; a step of a 784-1024-1024-10 classifier makes 66).  Function(address, kinds, types, slow) is called
 * like the ctypes function `slow`, whose kinds of arguments are given as text: P a pointer object of one of `types` or None, i a whole
 * number, f a float; other arguments, and signatures that are not in the table below, go to `slow`.  The interpreter's lock is
 * released during the call, as by ctypes.  kinds starting with v: a function without a result, which is None here too. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#define MAX_ARGS 12
#define MAX_TYPES 4

typedef union { void* p; int i; float f; } Arg;
typedef int (*Call)(void* fn, const Arg* a);

#define P_ void*
#define i_ int
#define f_ float
#define SIGNATURES(S)                                                                                                              \
  S(, "", (), ()) S(, "P", (P_), (a[0].p)) S(, "Pf", (P_, f_), (a[0].p, a[1].f)) S(, "Pi", (P_, i_), (a[0].p, a[1].i))             \
  S(, "PP", (P_, P_), (a[0].p, a[1].p)) S(, "PPP", (P_, P_, P_), (a[0].p, a[1].p, a[2].p))                                          \
  S(, "PPf", (P_, P_, f_), (a[0].p, a[1].p, a[2].f)) S(, "PfP", (P_, f_, P_), (a[0].p, a[1].f, a[2].p))                             \
  S(, "PPi", (P_, P_, i_), (a[0].p, a[1].p, a[2].i)) S(, "Pii", (P_, i_, i_), (a[0].p, a[1].i, a[2].i))                             \
  S(, "PPif", (P_, P_, i_, f_), (a[0].p, a[1].p, a[2].i, a[3].f)) S(, "PPff", (P_, P_, f_, f_), (a[0].p, a[1].p, a[2].f, a[3].f))   \
  S(, "PPii", (P_, P_, i_, i_), (a[0].p, a[1].p, a[2].i, a[3].i)) S(, "PPPf", (P_, P_, P_, f_), (a[0].p, a[1].p, a[2].p, a[3].f))   \
  S(, "PPPP", (P_, P_, P_, P_), (a[0].p, a[1].p, a[2].p, a[3].p))                                                                   \
  S(, "PPPff", (P_, P_, P_, f_, f_), (a[0].p, a[1].p, a[2].p, a[3].f, a[4].f))                                                      \
  S(, "PPPffffi", (P_, P_, P_, f_, f_, f_, f_, i_), (a[0].p, a[1].p, a[2].p, a[3].f, a[4].f, a[5].f, a[6].f, a[7].i))               \
  S(v, "vPPPiiiii", (P_, P_, P_, i_, i_, i_, i_, i_), (a[0].p, a[1].p, a[2].p, a[3].i, a[4].i, a[5].i, a[6].i, a[7].i))             \
  S(v, "vPPPiiiiiii", (P_, P_, P_, i_, i_, i_, i_, i_, i_, i_),                                                                     \
    (a[0].p, a[1].p, a[2].p, a[3].i, a[4].i, a[5].i, a[6].i, a[7].i, a[8].i, a[9].i))                                               \
  S(v, "vPPiiiii", (P_, P_, i_, i_, i_, i_, i_), (a[0].p, a[1].p, a[2].i, a[3].i, a[4].i, a[5].i, a[6].i))                          \
  S(v, "vPPPPiiii", (P_, P_, P_, P_, i_, i_, i_, i_), (a[0].p, a[1].p, a[2].p, a[3].p, a[4].i, a[5].i, a[6].i, a[7].i))             \
  S(v, "vPPPiiff", (P_, P_, P_, i_, i_, f_, f_), (a[0].p, a[1].p, a[2].p, a[3].i, a[4].i, a[5].f, a[6].f))                          \
  S(v, "vPPPPPiiff", (P_, P_, P_, P_, P_, i_, i_, f_, f_), (a[0].p, a[1].p, a[2].p, a[3].p, a[4].p, a[5].i, a[6].i, a[7].f, a[8].f))

#define RESULT_(types, args) return ((int (*) types)fn) args
#define RESULT_v(types, args) ((void (*) types)fn) args; return 0
/* (one function per signature, in the order of the table: call_1 ..) */
enum { BEFORE = __COUNTER__ };
_Static_assert(BEFORE == 0, "functions are numbered from 1");
#define DEFINE(V, kinds, types, args) DEFINE2(V, types, args, __COUNTER__)
#define DEFINE2(V, types, args, n) DEFINE3(V, types, args, n)
#define DEFINE3(V, types, args, n) static int call_##n(void* fn, const Arg* a) { (void)a; RESULT_##V(types, args); }
SIGNATURES(DEFINE)
#define KINDS(V, kinds, types, args) kinds,
static const char* const g_kinds[] = {SIGNATURES(KINDS)};
#define N_SIGNATURES (sizeof g_kinds / sizeof *g_kinds)
static const Call g_calls[] = {call_1, call_2, call_3, call_4, call_5, call_6, call_7, call_8, call_9, call_10, call_11, call_12, call_13,
                               call_14, call_15, call_16, call_17, call_18, call_19, call_20, call_21, call_22, call_23};
_Static_assert(sizeof g_calls / sizeof *g_calls == sizeof g_kinds / sizeof *g_kinds, "one function per signature");

typedef struct {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  void* fn;
  Call call;
  const char* kinds;
  int n, is_void;
  PyTypeObject* types[MAX_TYPES];
  PyObject* slow;
} Function;

static PyObject* function_call(PyObject* callable, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  Function* self = (Function*)callable;
  const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
  Arg a[MAX_ARGS];
  if (n != self->n || (kwnames && PyTuple_GET_SIZE(kwnames))) goto slow;
  for (int i = 0; i < self->n; ++i) {
    PyObject* o = args[i];
    if (self->kinds[i] == 'P') {
      if (o == Py_None) { a[i].p = NULL; continue; }
      int known = 0;
      for (int t = 0; t < MAX_TYPES; ++t) known |= self->types[t] && Py_TYPE(o) == self->types[t];
      Py_buffer view;
      if (!known) goto slow;
      if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) { PyErr_Clear(); goto slow; }
      if (view.len != (Py_ssize_t)sizeof(void*)) { PyBuffer_Release(&view); goto slow; }
      memcpy(&a[i].p, view.buf, sizeof(void*));          /* a pointer object holds the address */
      PyBuffer_Release(&view);
    } else if (self->kinds[i] == 'f') {
      if (!PyFloat_Check(o)) goto slow;
      a[i].f = (float)PyFloat_AS_DOUBLE(o);
    } else {
      if (!PyLong_Check(o)) goto slow;
      int over;
      const long long v = PyLong_AsLongLongAndOverflow(o, &over);
      if (over || v < INT32_MIN || v > INT32_MAX) goto slow;
      a[i].i = (int)v;
    }
  }
  {
    int res;
    Py_BEGIN_ALLOW_THREADS
    res = self->call(self->fn, a);
    Py_END_ALLOW_THREADS
    if (self->is_void) Py_RETURN_NONE;
    return PyLong_FromLong(res);
  }
slow:
  return PyObject_Vectorcall(self->slow, args, nargsf, kwnames);
}

static PyObject* function_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  unsigned long long address;
  const char* kinds;
  PyObject *types, *slow;
  (void)kw;
  if (!PyArg_ParseTuple(args, "KsO!O", &address, &kinds, &PyTuple_Type, &types, &slow)) return NULL;
  size_t s = 0;
  while (s < N_SIGNATURES && strcmp(g_kinds[s], kinds) != 0) ++s;
  if (s == N_SIGNATURES) { PyErr_Format(PyExc_KeyError, "no call of kind %s", kinds); return NULL; }
  Function* self = (Function*)type->tp_alloc(type, 0);
  if (!self) return NULL;
  self->vectorcall = function_call;
  self->fn = (void*)(uintptr_t)address;
  self->call = g_calls[s];
  self->is_void = kinds[0] == 'v';
  self->kinds = g_kinds[s] + self->is_void;
  self->n = (int)strlen(self->kinds);
  for (Py_ssize_t t = 0; t < PyTuple_GET_SIZE(types) && t < MAX_TYPES; ++t) {
    PyObject* o = PyTuple_GET_ITEM(types, t);
    if (PyType_Check(o)) { Py_INCREF(o); self->types[t] = (PyTypeObject*)o; }
  }
  Py_INCREF(slow);
  self->slow = slow;
  return (PyObject*)self;
}

/* (these live as long as the module that makes them) */
static void function_dealloc(PyObject* o) {
  Function* self = (Function*)o;
  for (int t = 0; t < MAX_TYPES; ++t) Py_XDECREF(self->types[t]);
  Py_XDECREF(self->slow);
  Py_TYPE(o)->tp_free(o);
}

/* restype, argtypes and the like are those of the ctypes function, which is also what ctypes takes as an argument (cast) */
static PyObject* function_getattro(PyObject* o, PyObject* name) {
  PyObject* slow = ((Function*)o)->slow;
  PyObject* res = PyObject_GenericGetAttr(o, name);
  if (res || !PyErr_ExceptionMatches(PyExc_AttributeError)) return res;
  PyErr_Clear();
  if (PyUnicode_CompareWithASCIIString(name, "_as_parameter_") == 0) { Py_INCREF(slow); return slow; }
  return PyObject_GetAttr(slow, name);
}
/* ... and once a program has set one, the calls go there */
static int function_setattro(PyObject* o, PyObject* name, PyObject* value) {
  ((Function*)o)->n = -1;
  return value ? PyObject_SetAttr(((Function*)o)->slow, name, value) : PyObject_DelAttr(((Function*)o)->slow, name);
}

static PyTypeObject FunctionType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "deepnet_amd._fastcall.Function",
    .tp_basicsize = sizeof(Function),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL,
    .tp_vectorcall_offset = offsetof(Function, vectorcall),
    .tp_call = PyVectorcall_Call,
    .tp_getattro = function_getattro,
    .tp_setattro = function_setattro,
    .tp_new = function_new,
    .tp_dealloc = function_dealloc,
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", NULL, -1, NULL, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__fastcall(void) {
  if (PyType_Ready(&FunctionType) < 0) return NULL;
  PyObject* m = PyModule_Create(&module);
  if (!m) return NULL;
  Py_INCREF(&FunctionType);
  if (PyModule_AddObject(m, "Function", (PyObject*)&FunctionType) < 0) { Py_DECREF(&FunctionType); Py_DECREF(m); return NULL; }
  return m;
}
