/* Host-side call path of the modules and the op, as a CPython extension.
 *
 * An eager call of a small linear is bound by the host: its kernel runs 5 to
 * 12 µs. Through ctypes (eleven converted arguments, a Python loop over the
 * member descriptors) and a Python walk over the module's buffers a call took
 * 14 µs to issue (7 µs with these objects, which do the same work in C).
 *
 *   Watch(buffers)          what a module's buffers were when its kernel view
 *                           was built: every name, data pointer and in-place
 *                           version; `unchanged(buffers)` compares them anew
 *                           on each call.
 *   GroupCall(...)          ssl_slr_forward_group with everything but x's and
 *                           the outputs' pointers fixed; the members are
 *                           copied for each call, so threads may share one,
 *                           and the GIL is released around the launch.
 *   OpCall(...)             ssl_bsr_addmm_inplace likewise, for calls the
 *                           streaming kernel runs.
 *
 * Nothing here links against torch or the HIP library: tensors are reached
 * through their Python methods, and the entry points' addresses are given.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <string.h>

#include "ssalaad_amd.h"

static PyObject *s_data_ptr, *s_version;

/* (data_ptr, _version) of a tensor; 0 on success. */
static int tensor_state(PyObject* t, unsigned long long* ptr, long long* version) {
  PyObject* v = PyObject_CallMethodNoArgs(t, s_data_ptr);
  if (!v) return -1;
  *ptr = PyLong_AsUnsignedLongLongMask(v);
  Py_DECREF(v);
  v = PyObject_GetAttr(t, s_version);
  if (!v) return -1;
  *version = PyLong_AsLongLong(v);
  Py_DECREF(v);
  return PyErr_Occurred() ? -1 : 0;
}

/* ------------------------------------------------------------------ Watch -- */
typedef struct {
  PyObject* name;
  int present;
  unsigned long long ptr;
  long long version;
} Item;

typedef struct {
  PyObject_HEAD
  Py_ssize_t n;
  Item* items;
} Watch;

static void watch_dealloc(Watch* w) {
  for (Py_ssize_t i = 0; i < w->n; ++i) Py_XDECREF(w->items[i].name);
  PyMem_Free(w->items);
  Py_TYPE(w)->tp_free((PyObject*)w);
}

static PyObject* watch_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  PyObject* d;
  if (kw || !PyArg_ParseTuple(args, "O!", &PyDict_Type, &d)) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "Watch takes one dict");
    return NULL;
  }
  Watch* w = (Watch*)type->tp_alloc(type, 0);
  if (!w) return NULL;
  /* a list of its own: a tensor's methods may change the dict */
  PyObject* pairs = PyDict_Items(d);
  const Py_ssize_t n = pairs ? PyList_GET_SIZE(pairs) : 0;
  w->items = pairs ? (Item*)PyMem_Calloc(n ? n : 1, sizeof(Item)) : NULL;
  if (!w->items) {
    if (pairs) PyErr_NoMemory();
    Py_XDECREF(pairs);
    Py_DECREF(w);
    return NULL;
  }
  while (w->n < n) {
    PyObject* pair = PyList_GET_ITEM(pairs, w->n);
    PyObject* t = PyTuple_GET_ITEM(pair, 1);
    Item* it = &w->items[w->n++];
    it->name = Py_NewRef(PyTuple_GET_ITEM(pair, 0));
    it->present = t != Py_None;
    if (it->present && tensor_state(t, &it->ptr, &it->version)) {
      Py_DECREF(pairs);
      Py_DECREF(w);
      return NULL;
    }
  }
  Py_DECREF(pairs);
  return (PyObject*)w;
}

static PyObject* watch_unchanged(Watch* w, PyObject* d) {
  if (!PyDict_Check(d)) {
    PyErr_SetString(PyExc_TypeError, "unchanged takes a dict");
    return NULL;
  }
  if (PyDict_Size(d) != w->n) Py_RETURN_FALSE;
  for (Py_ssize_t i = 0; i < w->n; ++i) {
    const Item* it = &w->items[i];
    PyObject* t = PyDict_GetItemWithError(d, it->name);
    if (!t) {
      if (PyErr_Occurred()) return NULL;
      Py_RETURN_FALSE;
    }
    if ((t != Py_None) != it->present) Py_RETURN_FALSE;
    if (!it->present) continue;
    unsigned long long ptr;
    long long version;
    Py_INCREF(t);
    const int bad = tensor_state(t, &ptr, &version);
    Py_DECREF(t);
    if (bad) return NULL;
    if (ptr != it->ptr || version != it->version) Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
}

static PyMethodDef watch_methods[] = {
    {"unchanged", (PyCFunction)watch_unchanged, METH_O,
     "whether every buffer still has its data pointer and version"},
    {NULL, NULL, 0, NULL}};

static PyTypeObject WatchType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "hostcall.Watch",
    .tp_basicsize = sizeof(Watch),
    .tp_flags = Py_TPFLAGS_DEFAULT,
    .tp_doc = "Data pointers and versions of a module's buffers",
    .tp_new = watch_new,
    .tp_dealloc = (destructor)watch_dealloc,
    .tp_methods = watch_methods,
};

/* -------------------------------------------------------------- GroupCall -- */
typedef int (*group_fn)(const void*, int64_t, int64_t, int64_t, int64_t, int32_t, int32_t, int32_t,
                        const ssl_slr_member*, int32_t, void*);

enum { MAX_MEMBERS = 4 };

typedef struct {
  PyObject_HEAD
  group_fn fn;
  const volatile uint64_t* status; /* host word: nonzero refuses the call */
  int64_t ldx, M, m, m_pad;
  int32_t p, q, dtype, n;
  void* stream;
  ssl_slr_member members[MAX_MEMBERS];
} GroupCall;

static PyObject* group_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  unsigned long long fn, status, members, stream;
  long long ldx, M, m, m_pad;
  int p, q, dtype, n;
  if (kw || !PyArg_ParseTuple(args, "KKLLLLiiiKiK", &fn, &status, &ldx, &M, &m, &m_pad, &p, &q,
                              &dtype, &members, &n, &stream)) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "GroupCall takes no keywords");
    return NULL;
  }
  if (!fn || !status || !members || n < 1 || n > MAX_MEMBERS) {
    PyErr_SetString(PyExc_ValueError, "GroupCall: bad arguments");
    return NULL;
  }
  GroupCall* g = (GroupCall*)type->tp_alloc(type, 0);
  if (!g) return NULL;
  g->fn = (group_fn)(uintptr_t)fn;
  g->status = (const volatile uint64_t*)(uintptr_t)status;
  g->ldx = ldx; g->M = M; g->m = m; g->m_pad = m_pad;
  g->p = p; g->q = q; g->dtype = dtype; g->n = n;
  g->stream = (void*)(uintptr_t)stream;
  memcpy(g->members, (const void*)(uintptr_t)members, sizeof(ssl_slr_member) * n);
  return (PyObject*)g;
}

/* launch(x, y...) -> the entry point's status, or −1 when an earlier call on
 * the device gave up a wait (nothing is launched then). */
static PyObject* group_launch(GroupCall* g, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != g->n + 1) {
    PyErr_Format(PyExc_TypeError, "launch takes x and %d outputs", (int)g->n);
    return NULL;
  }
  const unsigned long long x = PyLong_AsUnsignedLongLong(args[0]);
  ssl_slr_member mb[MAX_MEMBERS];
  memcpy(mb, g->members, sizeof(ssl_slr_member) * g->n);
  for (int i = 0; i < g->n; ++i) mb[i].y = (void*)(uintptr_t)PyLong_AsUnsignedLongLong(args[1 + i]);
  if (PyErr_Occurred()) return NULL;
  if (*g->status != 0) return PyLong_FromLong(-1);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g->fn((const void*)(uintptr_t)x, g->ldx, g->M, g->m, g->m_pad, g->p, g->q, g->dtype, mb, g->n,
             g->stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

static PyMethodDef group_methods[] = {
    {"launch", (PyCFunction)(void (*)(void))group_launch, METH_FASTCALL, "launch(x, y...)"},
    {NULL, NULL, 0, NULL}};

static void plain_dealloc(PyObject* o) { Py_TYPE(o)->tp_free(o); }

static PyTypeObject GroupCallType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "hostcall.GroupCall",
    .tp_basicsize = sizeof(GroupCall),
    .tp_flags = Py_TPFLAGS_DEFAULT,
    .tp_doc = "A fused call with its descriptors fixed",
    .tp_new = group_new,
    .tp_dealloc = plain_dealloc,
    .tp_methods = group_methods,
};

/* ----------------------------------------------------------------- OpCall -- */
typedef int (*op_fn)(void*, int64_t, const void*, int64_t, const int32_t*, const void*, int64_t,
                     const int32_t*, int64_t, int64_t, const void*, const int32_t*, const int32_t*,
                     int64_t, int32_t, int64_t, int64_t, int64_t, int64_t, int32_t, int32_t, int32_t,
                     int32_t*, int64_t, void*, int64_t, void*);

typedef struct {
  PyObject_HEAD
  op_fn fn;
  const volatile uint64_t* status; /* NULL: the device has no status word (yet) */
  int64_t ldo, ldx, nnz, n_chunks, n_slots, M, N, K, NB, n_counters, ws_bytes;
  int32_t p, q, dtype;
  const int32_t *col, *plan;
  int32_t* counters;
  void *ws, *stream;
} OpCall;

static PyObject* op_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  unsigned long long fn, status, col, plan, counters, ws, stream;
  long long ldo, ldx, nnz, n_chunks, n_slots, M, N, K, NB, n_counters, ws_bytes;
  int p, q, dtype;
  if (kw || !PyArg_ParseTuple(args, "KKLLKLKLLLLLLiiiKLKLK", &fn, &status, &ldo, &ldx, &col, &nnz,
                              &plan, &n_chunks, &n_slots, &M, &N, &K, &NB, &p, &q, &dtype,
                              &counters, &n_counters, &ws, &ws_bytes, &stream)) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "OpCall takes no keywords");
    return NULL;
  }
  if (!fn) {
    PyErr_SetString(PyExc_ValueError, "OpCall: bad arguments");
    return NULL;
  }
  OpCall* o = (OpCall*)type->tp_alloc(type, 0);
  if (!o) return NULL;
  o->fn = (op_fn)(uintptr_t)fn;
  o->status = (const volatile uint64_t*)(uintptr_t)status;
  o->ldo = ldo; o->ldx = ldx; o->nnz = nnz; o->n_chunks = n_chunks; o->n_slots = n_slots;
  o->M = M; o->N = N; o->K = K; o->NB = NB; o->n_counters = n_counters; o->ws_bytes = ws_bytes;
  o->p = p; o->q = q; o->dtype = dtype;
  o->col = (const int32_t*)(uintptr_t)col;
  o->plan = (const int32_t*)(uintptr_t)plan;
  o->counters = (int32_t*)(uintptr_t)counters;
  o->ws = (void*)(uintptr_t)ws;
  o->stream = (void*)(uintptr_t)stream;
  return (PyObject*)o;
}

/* launch(out, x, values): as GroupCall.launch. */
static PyObject* op_launch(OpCall* o, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3) {
    PyErr_SetString(PyExc_TypeError, "launch takes out, x and values");
    return NULL;
  }
  void* out = (void*)(uintptr_t)PyLong_AsUnsignedLongLong(args[0]);
  const void* x = (const void*)(uintptr_t)PyLong_AsUnsignedLongLong(args[1]);
  const void* values = (const void*)(uintptr_t)PyLong_AsUnsignedLongLong(args[2]);
  if (PyErr_Occurred()) return NULL;
  if (o->status && *o->status != 0) return PyLong_FromLong(-1);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = o->fn(out, o->ldo, x, o->ldx, o->col, values, o->nnz, o->plan, o->n_chunks, o->n_slots, NULL,
             NULL, NULL, 0, 0, o->M, o->N, o->K, o->NB, o->p, o->q, o->dtype, o->counters,
             o->n_counters, o->ws, o->ws_bytes, o->stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

static PyMethodDef op_methods[] = {
    {"launch", (PyCFunction)(void (*)(void))op_launch, METH_FASTCALL, "launch(out, x, values)"},
    {NULL, NULL, 0, NULL}};

static PyTypeObject OpCallType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "hostcall.OpCall",
    .tp_basicsize = sizeof(OpCall),
    .tp_flags = Py_TPFLAGS_DEFAULT,
    .tp_doc = "A streaming call of the in-place op with its structure fixed",
    .tp_new = op_new,
    .tp_dealloc = plain_dealloc,
    .tp_methods = op_methods,
};

static struct PyModuleDef module = {
    PyModuleDef_HEAD_INIT, "hostcall", "Host-side call path", -1, NULL, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit_hostcall(void) {
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  s_version = PyUnicode_InternFromString("_version");
  if (!s_data_ptr || !s_version || PyType_Ready(&WatchType) < 0 ||
      PyType_Ready(&GroupCallType) < 0 || PyType_Ready(&OpCallType) < 0)
    return NULL;
  PyObject* m = PyModule_Create(&module);
  if (!m) return NULL;
  if (PyModule_AddObjectRef(m, "Watch", (PyObject*)&WatchType) < 0 ||
      PyModule_AddObjectRef(m, "GroupCall", (PyObject*)&GroupCallType) < 0 ||
      PyModule_AddObjectRef(m, "OpCall", (PyObject*)&OpCallType) < 0 ||
      PyModule_AddIntConstant(m, "MEMBER_BYTES", (long)sizeof(ssl_slr_member)) < 0) {
    Py_DECREF(m);
    return NULL;
  }
  return m;
}
