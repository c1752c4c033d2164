/* The host mirror's native part: device blocks, arrays and calls of libknet8 as CPython objects.
 *
 * A training step of a small model is some twenty launches of 2 us each; as Python classes and ctypes calls the arrays and arguments around a launch took 10 us.
 * Here are KnetPtr (an owned or borrowed device block), ArrayBase (pointer, dims, element type; KnetArray derives from it) and Library, whose call() finds an entry
 * point by name, converts the arguments by its signature and appends the current stream.  What call() cannot convert it hands to `slow_call` (ctypes), which converts
 * or refuses it.  The global lock is released around every call into the library, as ctypes does. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>
#include <stdint.h>
#include <string.h>

typedef union { int i; long long l; unsigned long long u; float f; double d; void* p; char c; } Value;
#include "gen/knet8_calls_gen.h"   /* kSignatures, invoke() */

enum { kMaxArgs = 32 };

static void* (*g_malloc)(size_t) = NULL;
static void (*g_free)(void*) = NULL;
static PyObject* g_parked = NULL;        /* list that takes the blocks released while a launch sequence is captured, or NULL */
static PyObject* g_out_of_memory = NULL; /* raises */
static PyObject* g_dtype_class = NULL;   /* numpy.dtype */
static PyObject* g_dtypes[3];            /* float32, float64, int32 */
static PyObject* g_suffix[3];            /* "32", "64", None */
static const Py_ssize_t g_itemsize[3] = {4, 8, 4};
static PyTypeObject* g_array_type = NULL; /* KnetArray */
static PyObject* g_library = NULL;        /* the Library that knet8() calls */

/* ---- KnetPtr ------------------------------------------------------------------------------------------------------------------- */
typedef struct {
  PyObject_HEAD
  unsigned long long ptr;
  PyObject *nbytes, *keep, *weak;   /* keep None: the block is this object's and goes back to the pool with it */
} Ptr;
static PyTypeObject PtrType;

static size_t take_block(size_t nbytes) {
  void* p;
  if (!g_malloc) { PyErr_SetString(PyExc_RuntimeError, "libknet8 is not loaded"); return 0; }
  Py_BEGIN_ALLOW_THREADS
  p = g_malloc(nbytes ? nbytes : 1);
  Py_END_ALLOW_THREADS
  if (!p) {
    PyObject* r = PyObject_CallNoArgs(g_out_of_memory);
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_MemoryError, "Out of gpu memory");
  }
  return (size_t)p;
}

static int ptr_init(Ptr* s, PyObject* args, PyObject* kw) {
  static char* names[] = {"nbytes", "ptr", "keep", NULL};
  PyObject *nbytes = Py_None, *ptr = Py_None, *keep = Py_None;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "|OOO", names, &nbytes, &ptr, &keep)) return -1;
  if (s->keep) { PyErr_SetString(PyExc_RuntimeError, "KnetPtr is initialised once"); return -1; }
  if (ptr != Py_None) {   /* borrowed memory, kept alive through keep */
    PyObject* i = PyNumber_Long(ptr);
    if (!i) return -1;
    s->ptr = (size_t)PyLong_AsUnsignedLongLongMask(i);
    Py_DECREF(i);
    if (PyErr_Occurred()) return -1;
    Py_INCREF(nbytes); s->nbytes = nbytes;
    Py_INCREF(keep); s->keep = keep;
    return 0;
  }
  PyObject* n = PyNumber_Long(nbytes);
  if (!n) return -1;
  const long long want = PyLong_AsLongLong(n);
  if (want == -1 && PyErr_Occurred()) { Py_DECREF(n); return -1; }
  const size_t p = take_block(want > 0 ? (size_t)want : 0);
  if (!p) { Py_DECREF(n); return -1; }
  s->ptr = p;
  s->nbytes = n;
  Py_INCREF(Py_None); s->keep = Py_None;
  return 0;
}

static Ptr* ptr_new(size_t nbytes) {
  const size_t p = take_block(nbytes);
  if (!p) return NULL;
  Ptr* s = (Ptr*)PtrType.tp_alloc(&PtrType, 0);
  if (!s) { g_free((void*)p); return NULL; }
  s->ptr = p;
  s->nbytes = PyLong_FromSize_t(nbytes);
  Py_INCREF(Py_None); s->keep = Py_None;
  if (!s->nbytes) { Py_DECREF(s); return NULL; }
  return s;
}

static int ptr_traverse(Ptr* s, visitproc visit, void* arg) { Py_VISIT(s->nbytes); Py_VISIT(s->keep); return 0; }
static int ptr_clear(Ptr* s) {
  Py_CLEAR(s->nbytes);
  if (s->keep != Py_None) Py_CLEAR(s->keep);   /* (None says whose the block is, until the end) */
  return 0;
}

static void ptr_dealloc(Ptr* s) {
  PyObject_GC_UnTrack(s);
  if (s->weak) PyObject_ClearWeakRefs((PyObject*)s);
  if (s->ptr && s->keep == Py_None) {
    int parked = 0;
    if (g_parked) {
      PyObject *t, *v, *tb;
      PyErr_Fetch(&t, &v, &tb);
      PyObject* o = PyLong_FromUnsignedLongLong(s->ptr);
      parked = o && PyList_Append(g_parked, o) == 0;
      Py_XDECREF(o);
      PyErr_Restore(t, v, tb);
    }
    if (!parked && g_free) g_free((void*)(size_t)s->ptr);
  }
  ptr_clear(s);
  Py_CLEAR(s->keep);
  Py_TYPE(s)->tp_free((PyObject*)s);
}

static PyMemberDef ptr_members[] = {{"ptr", T_ULONGLONG, offsetof(Ptr, ptr), 0, "device address"},
                                    {"nbytes", T_OBJECT, offsetof(Ptr, nbytes), 0, "size in bytes"},
                                    {"_keep", T_OBJECT, offsetof(Ptr, keep), 0, "owner of borrowed memory; None: the block belongs to this object"},
                                    {NULL}};
static PyTypeObject PtrType = {PyVarObject_HEAD_INIT(NULL, 0).tp_name = "knet8.KnetPtr",
                               .tp_doc = "Owner of one device allocation (src/knetarrays/kptr.jl:10-15), or a borrowed address and what keeps it alive.",
                               .tp_basicsize = sizeof(Ptr), .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC, .tp_new = PyType_GenericNew,
                               .tp_init = (initproc)ptr_init, .tp_dealloc = (destructor)ptr_dealloc, .tp_traverse = (traverseproc)ptr_traverse,
                               .tp_clear = (inquiry)ptr_clear, .tp_weaklistoffset = offsetof(Ptr, weak), .tp_members = ptr_members};

/* ---- ArrayBase ----------------------------------------------------------------------------------------------------------------- */
typedef struct {
  PyObject_HEAD
  Ptr* kptr;
  PyObject *dims, *dtype;   /* tuple of int; numpy dtype */
  int type;                 /* index into g_suffix; kOther: no kernels for it */
  Py_ssize_t itemsize, offset, length;
} Array;
enum { kOther = 2 };
static PyTypeObject ArrayType;

/* The dtype object for what the caller named (a new reference): one of the three, or what numpy makes of it.  numpy has several objects for one type (every dtype that comes
 * out of a pickle is a new one, and what is made of such an array carries it on): they count as the one they are equal to. */
static PyObject* as_dtype(PyObject* d, int* type, Py_ssize_t* itemsize) {
  for (int i = 0; i < 3; i++)
    if (d == g_dtypes[i]) { *type = i; *itemsize = g_itemsize[i]; Py_INCREF(d); return d; }
  PyObject* n = PyObject_CallFunctionObjArgs(g_dtype_class, d, NULL);
  if (!n) return NULL;
  for (int i = 0; i < 3; i++) {
    const int same = n == g_dtypes[i] ? 1 : PyObject_RichCompareBool(n, g_dtypes[i], Py_EQ);
    if (same < 0) { Py_DECREF(n); return NULL; }
    if (same) { *type = i; *itemsize = g_itemsize[i]; Py_INCREF(g_dtypes[i]); Py_DECREF(n); return g_dtypes[i]; }
  }
  PyObject* size = PyObject_GetAttrString(n, "itemsize");
  *itemsize = size ? PyLong_AsSsize_t(size) : -1;
  *type = kOther;
  Py_XDECREF(size);
  if (PyErr_Occurred()) Py_CLEAR(n);
  return n;
}

/* A tuple of ints of any sequence of numbers (a new reference) and their product. */
static PyObject* as_dims(PyObject* o, Py_ssize_t* length) {
  PyObject* seq = PySequence_Tuple(o);
  if (!seq) return NULL;
  const Py_ssize_t n = PyTuple_GET_SIZE(seq);
  int exact = 1;
  for (Py_ssize_t i = 0; i < n; i++) exact = exact && PyLong_CheckExact(PyTuple_GET_ITEM(seq, i));
  if (!exact) {
    PyObject* t = PyTuple_New(n);
    for (Py_ssize_t i = 0; t && i < n; i++) {
      PyObject* v = PyNumber_Long(PyTuple_GET_ITEM(seq, i));
      if (!v) { Py_CLEAR(t); break; }
      PyTuple_SET_ITEM(t, i, v);
    }
    Py_DECREF(seq);
    if (!t) return NULL;
    seq = t;
  }
  Py_ssize_t len = 1;
  for (Py_ssize_t i = 0; i < n; i++) {
    const Py_ssize_t d = PyLong_AsSsize_t(PyTuple_GET_ITEM(seq, i));
    if (d == -1 && PyErr_Occurred()) { Py_DECREF(seq); return NULL; }
    if (__builtin_mul_overflow(len, d, &len)) {
      PyErr_SetString(PyExc_OverflowError, "array too large");
      Py_DECREF(seq);
      return NULL;
    }
  }
  *length = len;
  return seq;
}

static PyObject* array_new(PyTypeObject* t, PyObject* args, PyObject* kw) {
  (void)args; (void)kw;
  return t->tp_alloc(t, 0);
}

/* _init(kptr or None, dims, dtype, offset): a view of kptr, or a block of its own */
static PyObject* array_init(Array* s, PyObject* args) {
  PyObject *k, *dims, *dtype;
  Py_ssize_t offset = 0, length = 0;
  if (!PyArg_ParseTuple(args, "OOO|n", &k, &dims, &dtype, &offset)) return NULL;
  if (k != Py_None && !PyObject_TypeCheck(k, &PtrType)) { PyErr_SetString(PyExc_TypeError, "a KnetPtr is needed"); return NULL; }
  int type;
  Py_ssize_t itemsize;
  PyObject *t = as_dtype(dtype, &type, &itemsize), *d = t ? as_dims(dims, &length) : NULL;
  if (d && k == Py_None) k = (PyObject*)ptr_new(length > 0 ? (size_t)length * itemsize : 0);
  else Py_INCREF(k);
  if (!d || !k) { Py_XDECREF(t); Py_XDECREF(d); Py_XDECREF(k); return NULL; }
  s->type = type; s->itemsize = itemsize; s->offset = offset; s->length = length;
  Py_XSETREF(s->kptr, (Ptr*)k);
  Py_XSETREF(s->dims, d);
  Py_XSETREF(s->dtype, t);
  Py_RETURN_NONE;
}

/* takes over kptr, dims and dtype */
static Array* array_make(Ptr* kptr, PyObject* dims, PyObject* dtype, int type, Py_ssize_t itemsize, Py_ssize_t offset, Py_ssize_t length) {
  Array* a = kptr && dims ? (Array*)g_array_type->tp_alloc(g_array_type, 0) : NULL;
  if (!a) { Py_XDECREF(kptr); Py_XDECREF(dims); Py_XDECREF(dtype); return NULL; }
  a->kptr = kptr; a->dims = dims; a->dtype = dtype; a->type = type; a->itemsize = itemsize; a->offset = offset; a->length = length;
  return a;
}

static int ready(Array* s) {
  if (s->dtype && s->kptr && s->dims) return 1;
  PyErr_SetString(PyExc_RuntimeError, "KnetArray is not initialised");
  return 0;
}

/* similar(dims=None, dtype=None) */
static PyObject* array_similar(Array* s, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  PyObject *dims = Py_None, *dtype = Py_None;
  const Py_ssize_t nkw = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  if (nargs > 2) { PyErr_SetString(PyExc_TypeError, "similar(dims=None, dtype=None)"); return NULL; }
  if (nargs > 0) dims = args[0];
  if (nargs > 1) dtype = args[1];
  for (Py_ssize_t i = 0; i < nkw; i++) {
    PyObject* n = PyTuple_GET_ITEM(kwnames, i);
    if (PyUnicode_CompareWithASCIIString(n, "dims") == 0 && nargs < 1) dims = args[nargs + i];
    else if (PyUnicode_CompareWithASCIIString(n, "dtype") == 0 && nargs < 2) dtype = args[nargs + i];
    else { PyErr_Format(PyExc_TypeError, "similar() got an unexpected keyword argument %R", n); return NULL; }
  }
  if (!ready(s)) return NULL;
  int type = s->type;
  Py_ssize_t length = s->length, itemsize = s->itemsize;
  PyObject *d = s->dims, *t = s->dtype;
  if (dtype == Py_None) Py_INCREF(t);
  else if (!(t = as_dtype(dtype, &type, &itemsize))) return NULL;
  if (dims == Py_None) Py_INCREF(d);
  else if (!(d = as_dims(dims, &length))) { Py_DECREF(t); return NULL; }
  return (PyObject*)array_make(ptr_new(length > 0 ? (size_t)length * itemsize : 0), d, t, type, itemsize, 0, length);
}

/* _view(dims, offset): other dims over the same memory, offset bytes from its start */
static PyObject* array_view(Array* s, PyObject* const* args, Py_ssize_t nargs) {
  Py_ssize_t length = 0;
  if (!ready(s)) return NULL;
  Py_ssize_t offset = s->offset;
  if (nargs < 1 || nargs > 2) { PyErr_SetString(PyExc_TypeError, "_view(dims, offset)"); return NULL; }
  if (nargs == 2) {
    offset = PyLong_AsSsize_t(args[1]);
    if (offset == -1 && PyErr_Occurred()) return NULL;
  }
  PyObject* d = as_dims(args[0], &length);
  if (!d) return NULL;
  Py_INCREF(s->kptr);
  Py_INCREF(s->dtype);
  return (PyObject*)array_make(s->kptr, d, s->dtype, s->type, s->itemsize, offset, length);
}

/* size() -> dims; size(i) -> the i-th, 1 beyond the last */
static PyObject* array_size(Array* s, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  PyObject* i = Py_None;
  if (!ready(s)) return NULL;
  if (nargs == 1 && !kwnames) i = args[0];
  else if (nargs == 0 && kwnames && PyTuple_GET_SIZE(kwnames) == 1 && PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(kwnames, 0), "i") == 0) i = args[0];
  else if (nargs != 0 || kwnames) { PyErr_SetString(PyExc_TypeError, "size(i=None)"); return NULL; }
  if (i == Py_None) { Py_INCREF(s->dims); return s->dims; }
  Py_ssize_t k = PyNumber_AsSsize_t(i, PyExc_IndexError);
  if (k == -1 && PyErr_Occurred()) return NULL;
  const Py_ssize_t nd = PyTuple_GET_SIZE(s->dims);
  if (k > nd) return PyLong_FromLong(1);
  k = k >= 1 ? k - 1 : k - 1 + nd;   /* (as an index of the tuple) */
  if (k < 0) { PyErr_SetString(PyExc_IndexError, "tuple index out of range"); return NULL; }
  PyObject* v = PyTuple_GET_ITEM(s->dims, k);
  Py_INCREF(v);
  return v;
}

/* stride(i): elements from one index of dimension i to the next */
static PyObject* array_stride(Array* s, PyObject* arg) {
  if (!ready(s)) return NULL;
  const Py_ssize_t i = PyNumber_AsSsize_t(arg, PyExc_IndexError);
  if (i == -1 && PyErr_Occurred()) return NULL;
  Py_ssize_t n = PyTuple_GET_SIZE(s->dims), st = 1, last = i - 1;
  if (last < 0) last = last + n < 0 ? 0 : last + n;   /* (as the end of a slice of the tuple) */
  for (Py_ssize_t k = 0; k < n && k < last; k++) st *= PyLong_AsSsize_t(PyTuple_GET_ITEM(s->dims, k));
  return PyLong_FromSsize_t(st);
}

static PyObject* array_get_ptr(Array* s, void* c) { (void)c; return ready(s) ? PyLong_FromUnsignedLongLong((unsigned long long)s->kptr->ptr + (unsigned long long)s->offset) : NULL; }
static PyObject* array_get_ndims(Array* s, void* c) { (void)c; return ready(s) ? PyLong_FromSsize_t(PyTuple_GET_SIZE(s->dims)) : NULL; }
static PyObject* array_get_suffix(Array* s, void* c) { (void)c; if (!ready(s)) return NULL; Py_INCREF(g_suffix[s->type]); return g_suffix[s->type]; }

static PyObject* array_get_dims(Array* s, void* c) { (void)c; if (!ready(s)) return NULL; Py_INCREF(s->dims); return s->dims; }
static int array_set_dims(Array* s, PyObject* v, void* c) {
  (void)c;
  Py_ssize_t length = 0;
  if (!v) { PyErr_SetString(PyExc_AttributeError, "dims cannot be deleted"); return -1; }
  PyObject* d = as_dims(v, &length);
  if (!d) return -1;
  s->length = length;
  Py_XSETREF(s->dims, d);
  return 0;
}

/* kptr and dtype are members, which read fastest; they are set here, so that what goes with them is too. */
static int array_setattro(PyObject* o, PyObject* name, PyObject* v) {
  Array* s = (Array*)o;
  if (v && PyUnicode_Check(name) && PyUnicode_CompareWithASCIIString(name, "dtype") == 0) {   /* other elements in the same memory */
    int type;
    Py_ssize_t itemsize;
    PyObject* t = as_dtype(v, &type, &itemsize);
    if (!t) return -1;
    s->type = type; s->itemsize = itemsize;
    Py_XSETREF(s->dtype, t);
    return 0;
  }
  if (v && PyUnicode_Check(name) && PyUnicode_CompareWithASCIIString(name, "kptr") == 0) {   /* other memory; offset stays */
    if (!PyObject_TypeCheck(v, &PtrType)) { PyErr_SetString(PyExc_TypeError, "a KnetPtr is needed"); return -1; }
    Py_INCREF(v);
    Py_XSETREF(s->kptr, (Ptr*)v);
    return 0;
  }
  return PyObject_GenericSetAttr(o, name, v);
}

static int array_traverse(Array* s, visitproc visit, void* arg) { Py_VISIT(s->kptr); Py_VISIT(s->dims); Py_VISIT(s->dtype); return 0; }
static int array_clear(Array* s) { Py_CLEAR(s->kptr); Py_CLEAR(s->dims); Py_CLEAR(s->dtype); return 0; }
static void array_dealloc(Array* s) {
  PyObject_GC_UnTrack(s);
  array_clear(s);
  Py_TYPE(s)->tp_free((PyObject*)s);
}

static PyMethodDef array_methods[] = {
    {"_init", (PyCFunction)array_init, METH_VARARGS, "_init(kptr, dims, dtype, offset=0)"},
    {"_view", (PyCFunction)(void*)array_view, METH_FASTCALL, "_view(dims, offset): the same memory under other dims"},
    {"similar", (PyCFunction)(void*)array_similar, METH_FASTCALL | METH_KEYWORDS,
     "``similar(x, dims)`` (src/knetarrays/abstractarray.jl:13-35): uninitialised array of the same kind."},
    {"size", (PyCFunction)(void*)array_size, METH_FASTCALL | METH_KEYWORDS, "size(x) and size(x, i)"},
    {"stride", (PyCFunction)array_stride, METH_O, "stride(x, i) in elements"},
    {NULL}};
static PyMemberDef array_members[] = {{"kptr", T_OBJECT_EX, offsetof(Array, kptr), READONLY, "the block"},
                                      {"dtype", T_OBJECT_EX, offsetof(Array, dtype), READONLY, "element type"},
                                      {"offset", T_PYSSIZET, offsetof(Array, offset), 0, "bytes from the start of the block"},
                                      {"length", T_PYSSIZET, offsetof(Array, length), READONLY, "number of elements"},
                                      {NULL}};
static PyGetSetDef array_getset[] = {{"ptr", (getter)array_get_ptr, NULL, "device address of the first element", NULL},
                                     {"ndims", (getter)array_get_ndims, NULL, "number of dimensions", NULL},
                                     {"dims", (getter)array_get_dims, (setter)array_set_dims, "Julia dims: the first varies fastest in memory", NULL},
                                     {"suffix", (getter)array_get_suffix, NULL, "\"32\" or \"64\": the element type in the names of entry points; None for Int32", NULL},
                                     {NULL}};
static PyTypeObject ArrayType = {PyVarObject_HEAD_INIT(NULL, 0).tp_name = "knet8.ArrayBase",
                                 .tp_doc = "Storage side of KnetArray: block, dims, element type.",
                                 .tp_basicsize = sizeof(Array), .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC, .tp_new = array_new,
                                 .tp_dealloc = (destructor)array_dealloc, .tp_traverse = (traverseproc)array_traverse, .tp_clear = (inquiry)array_clear,
                                 .tp_setattro = array_setattro, .tp_methods = array_methods, .tp_members = array_members, .tp_getset = array_getset};

/* ---- Library ------------------------------------------------------------------------------------------------------------------- */
typedef struct {
  PyObject_HEAD
  PyObject* entries;   /* dict: name without _stream -> capsule of Entry */
  PyObject* stream;    /* None (the null stream) or a handle */
} Library;
typedef struct { void* fn; int sig, nargs; const char* code; } Entry;   /* code: the return type, then the arguments */
static PyTypeObject LibraryType;

static void entry_free(PyObject* cap) { PyMem_Free(PyCapsule_GetPointer(cap, NULL)); }

/* _bind(name, address, signature): signature as in kSignatures, the stream's p last.  False if the generated table does not know it (call() then leaves it to slow_call). */
static PyObject* library_bind(Library* s, PyObject* args) {
  PyObject* name;
  unsigned long long addr;
  const char* code;
  if (!PyArg_ParseTuple(args, "UKs", &name, &addr, &code)) return NULL;
  int sig = -1;
  for (int i = 0; i < (int)(sizeof(kSignatures) / sizeof(kSignatures[0])); i++)
    if (strcmp(kSignatures[i], code) == 0) sig = i;
  const size_t n = strlen(code);
  if (sig < 0 || n < 2 || n > kMaxArgs || code[n - 1] != 'p') Py_RETURN_FALSE;
  Entry* e = (Entry*)PyMem_Malloc(sizeof(Entry));
  if (!e) return PyErr_NoMemory();
  e->fn = (void*)(size_t)addr; e->sig = sig; e->nargs = (int)n - 2; e->code = kSignatures[sig];
  PyObject* cap = PyCapsule_New(e, NULL, entry_free);
  if (!cap) { PyMem_Free(e); return NULL; }
  if (!s->entries) s->entries = PyDict_New();
  const int rc = s->entries ? PyDict_SetItem(s->entries, name, cap) : -1;
  Py_DECREF(cap);
  if (rc != 0) return NULL;
  Py_RETURN_TRUE;
}

/* 1: converted, 0: not a form that is converted here */
static int convert(PyObject* o, char code, Value* v) {
  switch (code) {
    case 'p':
      if (PyLong_CheckExact(o)) { v->u = PyLong_AsUnsignedLongLongMask(o); break; }
      if (o == Py_None) { v->p = NULL; break; }
      return 0;
    case 'i':
      if (!PyLong_CheckExact(o)) return 0;
      v->i = (int)PyLong_AsUnsignedLongMask(o);
      break;
    case 'l': case 'u':
      if (!PyLong_CheckExact(o)) return 0;
      v->u = PyLong_AsUnsignedLongLongMask(o);
      break;
    case 'f': case 'd': {
      double d;
      if (PyFloat_Check(o)) d = PyFloat_AS_DOUBLE(o);
      else if (Py_TYPE(o)->tp_as_number && Py_TYPE(o)->tp_as_number->nb_float) d = PyFloat_AsDouble(o);
      else return 0;
      if (code == 'f') v->f = (float)d;
      else v->d = d;
      break;
    }
    case 'c':
      if (!PyBytes_Check(o) || PyBytes_GET_SIZE(o) != 1) return 0;
      v->c = PyBytes_AS_STRING(o)[0];
      break;
    default: return 0;
  }
  if (PyErr_Occurred()) { PyErr_Clear(); return 0; }
  return 1;
}

static PyObject* library_call(Library* s, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs < 1) { PyErr_SetString(PyExc_TypeError, "call(fun, *args)"); return NULL; }
  PyObject* cap = s->entries ? PyDict_GetItemWithError(s->entries, args[0]) : NULL;
  if (!cap && PyErr_Occurred()) return NULL;
  Value v[kMaxArgs], r;
  const Entry* e = cap ? (const Entry*)PyCapsule_GetPointer(cap, NULL) : NULL;
  int fits = e != NULL && e->nargs == nargs - 1;
  for (Py_ssize_t i = 1; fits && i < nargs; i++) fits = convert(args[i], e->code[i], &v[i - 1]);
  if (fits) fits = convert(s->stream ? s->stream : Py_None, 'p', &v[nargs - 1]);
  if (!fits) {
    PyObject* slow = PyObject_GetAttrString((PyObject*)s, "slow_call");
    if (!slow) return NULL;
    PyObject* out = PyObject_Vectorcall(slow, args, nargs, NULL);
    Py_DECREF(slow);
    return out;
  }
  Py_BEGIN_ALLOW_THREADS
  invoke(e->sig, e->fn, v, &r);
  Py_END_ALLOW_THREADS
  switch (e->code[0]) {
    case 'i': return PyLong_FromLong(r.i);
    case 'f': return PyFloat_FromDouble(r.f);
    case 'd': return PyFloat_FromDouble(r.d);
    default: Py_RETURN_NONE;
  }
}

static int library_traverse(Library* s, visitproc visit, void* arg) { Py_VISIT(s->entries); Py_VISIT(s->stream); return 0; }
static int library_clear(Library* s) { Py_CLEAR(s->entries); Py_CLEAR(s->stream); return 0; }
static void library_dealloc(Library* s) {
  PyObject_GC_UnTrack(s);
  library_clear(s);
  Py_TYPE(s)->tp_free((PyObject*)s);
}
static PyMethodDef library_methods[] = {
    {"_bind", (PyCFunction)library_bind, METH_VARARGS, "_bind(name, address, signature)"},
    {"call", (PyCFunction)(void*)library_call, METH_FASTCALL, "``@knet8(fun, ...)``: asynchronous launch of ``<fun>_stream`` on the current stream."},
    {NULL}};
static PyMemberDef library_members[] = {{"stream", T_OBJECT, offsetof(Library, stream), 0, "current stream handle (None: the null stream), cf. CUDA.stream() in the reference"}, {NULL}};
static PyTypeObject LibraryType = {PyVarObject_HEAD_INIT(NULL, 0).tp_name = "knet8.Library", .tp_doc = "Calls entry points of libknet8 by name.",
                                   .tp_basicsize = sizeof(Library), .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC, .tp_new = PyType_GenericNew,
                                   .tp_dealloc = (destructor)library_dealloc, .tp_traverse = (traverseproc)library_traverse, .tp_clear = (inquiry)library_clear,
                                   .tp_methods = library_methods, .tp_members = library_members};

/* ---- module --------------------------------------------------------------------------------------------------------------------- */
static PyObject* mod_park(PyObject* m, PyObject* list) {
  (void)m;
  if (list != Py_None && !PyList_Check(list)) { PyErr_SetString(PyExc_TypeError, "park(list or None)"); return NULL; }
  PyObject* old = g_parked;
  g_parked = list == Py_None ? NULL : list;
  Py_XINCREF(g_parked);
  Py_XDECREF(old);
  Py_RETURN_NONE;
}

/* setup(malloc address, free address, out_of_memory, numpy.dtype, dtypes, library) */
static PyObject* mod_setup(PyObject* m, PyObject* args) {
  (void)m;
  unsigned long long a, f;
  PyObject *oom, *cls, *d0, *d1, *d2, *lib;
  if (!PyArg_ParseTuple(args, "KKOO(OOO)O!", &a, &f, &oom, &cls, &d0, &d1, &d2, &LibraryType, &lib)) return NULL;
  Py_INCREF(cls); Py_XSETREF(g_dtype_class, cls);
  PyObject* d[3] = {d0, d1, d2};
  for (int i = 0; i < 3; i++) { Py_INCREF(d[i]); Py_XSETREF(g_dtypes[i], d[i]); }
  Py_INCREF(oom); Py_XSETREF(g_out_of_memory, oom);
  Py_INCREF(lib); Py_XSETREF(g_library, lib);
  g_malloc = (void* (*)(size_t))(size_t)a;
  g_free = (void (*)(void*))(size_t)f;
  Py_RETURN_NONE;
}

static PyObject* mod_array_type(PyObject* m, PyObject* t) {
  (void)m;
  if (!PyType_Check(t) || !PyType_IsSubtype((PyTypeObject*)t, &ArrayType)) { PyErr_SetString(PyExc_TypeError, "a subclass of ArrayBase is needed"); return NULL; }
  Py_INCREF(t);
  Py_XSETREF(g_array_type, (PyTypeObject*)t);
  Py_RETURN_NONE;
}

static PyObject* mod_knet8(PyObject* m, PyObject* const* args, Py_ssize_t nargs) {
  (void)m;
  if (!g_library) { PyErr_SetString(PyExc_RuntimeError, "libknet8 is not loaded"); return NULL; }
  return library_call((Library*)g_library, args, nargs);
}

static PyMethodDef mod_methods[] = {{"park", mod_park, METH_O, "park(list): blocks that are released go into the list; park(None): back to the pool"},
                                    {"setup", mod_setup, METH_VARARGS, "setup(malloc, free, out_of_memory, dtype, dtypes, library)"},
                                    {"array_type", mod_array_type, METH_O, "array_type(cls): the class similar() and _view() make"},
                                    {"knet8", (PyCFunction)(void*)mod_knet8, METH_FASTCALL, "knet8(fun, *args): the loaded library's call()"},
                                    {NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_knet8_host", "Native part of the host mirror", -1, mod_methods};

#ifndef KNET8_BUILD_ID
#define KNET8_BUILD_ID "unknown"
#endif
PyMODINIT_FUNC PyInit__knet8_host(void) {
  if (PyType_Ready(&PtrType) < 0 || PyType_Ready(&ArrayType) < 0 || PyType_Ready(&LibraryType) < 0) return NULL;
  PyObject* m = PyModule_Create(&module);
  if (!m) return NULL;
  g_suffix[0] = PyUnicode_InternFromString("32");
  g_suffix[1] = PyUnicode_InternFromString("64");
  Py_INCREF(Py_None);
  g_suffix[2] = Py_None;
  Py_INCREF(&PtrType); Py_INCREF(&ArrayType); Py_INCREF(&LibraryType);
  if (!g_suffix[0] || !g_suffix[1] || PyModule_AddObject(m, "KnetPtr", (PyObject*)&PtrType) < 0 || PyModule_AddObject(m, "ArrayBase", (PyObject*)&ArrayType) < 0 ||
      PyModule_AddObject(m, "Library", (PyObject*)&LibraryType) < 0 || PyModule_AddStringConstant(m, "build_id", KNET8_BUILD_ID) < 0) {
    Py_DECREF(m);
    return NULL;
  }
  return m;
}
