// The call path of the Python front end: entry points called through a vectorcall object instead of ctypes, memory handles the garbage
// collector does not see, and the error check behind every call.
//
// A program of small operators (a TreeLSTM pass: 2300 calls, 0.6 ms of device work) is bound by its interpreter: a ctypes call costs 0.6 to
// 1.2 us, of which the entry point itself takes 0.1 to 0.2; a Python object with __slots__ 0.3 us, and each of the 17 objects that the
// collector followed per operator brings its full collections (20 ms beside a large library) closer.
//
// A call whose arguments are the ordinary ones (int, float, None, a ctypes array) is converted here, everything else goes to the ctypes
// function, which converts it or raises what it always raised.  The interpreter lock is released around the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <cstddef>
#include <cstdint>
#include <cstring>
#include <string>
#include <tuple>
#include <type_traits>
#include <utility>

namespace {
PyObject* g_array_type = nullptr;        // ctypes.Array

// ---- arguments: what ctypes' from_param gives for the same object; false: not an ordinary one -------------------------------------
inline bool convert(PyObject* o, void*& out) {
  if (PyLong_Check(o)) { out = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(o); return true; }
  if (o == Py_None) { out = nullptr; return true; }
  if (!PyObject_TypeCheck(o, (PyTypeObject*)g_array_type)) return false;
  Py_buffer view;
  if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) { PyErr_Clear(); return false; }
  out = view.buf;
  PyBuffer_Release(&view);               // (the caller of the call holds the array)
  return true;
}
inline bool convert(PyObject* o, int& out) { if (!PyLong_Check(o)) return false; out = (int)PyLong_AsUnsignedLongMask(o); return true; }
inline bool convert(PyObject* o, int64_t& out) { if (!PyLong_Check(o)) return false; out = (int64_t)PyLong_AsUnsignedLongLongMask(o); return true; }
inline bool convert(PyObject* o, size_t& out) { if (!PyLong_Check(o)) return false; out = (size_t)PyLong_AsUnsignedLongLongMask(o); return true; }
inline bool convert(PyObject* o, float& out) {
  if (PyFloat_Check(o)) { out = (float)PyFloat_AS_DOUBLE(o); return true; }
  if (!PyLong_Check(o)) return false;
  const double d = PyLong_AsDouble(o);
  if (d == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
  out = (float)d;
  return true;
}

// ---- one entry point ------------------------------------------------------------------------------------------------------------
struct Call;
typedef PyObject* (*Invoke)(Call*, PyObject* const*, bool&);
struct Call {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  void* fn;
  PyObject* fallback;                    // the ctypes function
  Invoke invoke;
  Py_ssize_t nargs;
};
template <class R> struct Result;
template <> struct Result<void*> { static PyObject* of(void* p) { if (!p) Py_RETURN_NONE; return PyLong_FromVoidPtr(p); } };
template <> struct Result<size_t> { static PyObject* of(size_t v) { return PyLong_FromSize_t(v); } };

template <class R, class... A, size_t... K>
PyObject* invoke_with(Call* c, PyObject* const* args, bool& ordinary, std::index_sequence<K...>) {
  std::tuple<A...> v;
  ordinary = (convert(args[K], std::get<K>(v)) && ...);
  if (!ordinary) return nullptr;
  R (*fn)(A...) = (R (*)(A...))c->fn;
  if constexpr (std::is_void<R>::value) {
    Py_BEGIN_ALLOW_THREADS
    fn(std::get<K>(v)...);
    Py_END_ALLOW_THREADS
    Py_RETURN_NONE;
  } else {
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = fn(std::get<K>(v)...);
    Py_END_ALLOW_THREADS
    return Result<R>::of(r);
  }
}
template <class R, class... A>
PyObject* invoke_as(Call* c, PyObject* const* args, bool& ordinary) { return invoke_with<R, A...>(c, args, ordinary, std::index_sequence_for<A...>()); }

template <class T> constexpr char letter() {
  return std::is_void<T>::value ? 'v' : std::is_same<T, void*>::value ? 'P' : std::is_same<T, int>::value ? 'I' : std::is_same<T, float>::value ? 'F' : std::is_same<T, int64_t>::value ? 'L' : 'Z';
}
struct Form { std::string name; Invoke invoke; };
template <class R, class... A> Form form() { return {std::string{letter<R>(), letter<A>()...}, &invoke_as<R, A...>}; }

// The signatures of the operators' entry points (what waits for the device or is called once stays with ctypes).
Invoke find_form(const char* name) {
  using P = void*; using I = int; using F = float; using L = int64_t; using Z = size_t; using V = void;
  static const Form forms[] = {
      form<P, Z>(), form<Z>(), form<V, Z>(), form<V>(), form<V, P, P, Z>(),
      form<V, P, F, L>(), form<V, P, P, L>(), form<V, P, P, F, L>(), form<V, P, F, P, F, P, L>(), form<V, P, P, P, L>(), form<V, P, P, P, F, P, F, L>(),
      form<V, I, P, P, L, F, F>(), form<V, I, P, P, P, P, L, I, F, F>(), form<V, I, P, P, F, L>(),
      form<V, I, P, P, P, P, P, P, I>(), form<V, I, P, P, P, I, P, P, P, I, P, P, I>(), form<V, I, P, P, P, P, I>(),
      form<V, I, I, I, F, P, I, P, F, P>(), form<V, I, I, I, I, I, F, P, I, P, I, F, P, I>(), form<V, I, I, P, P, P>(), form<V, P, P, P, I>(),
      form<V, P, P, I, I>(), form<V, P, P, I, I, I>(), form<V, P, P, P, P, I>(), form<V, P, P, P, I, I>(), form<V, I, P, P, I, I, I>(), form<V, I, P, P, P, I, I, I>(),
      form<V, I, P, P, P, I, I>(), form<V, I, P, P, P, P, I, I>(),
      form<V, P, P, P, P, I, I, I, I, I, I, I, I, I, I, I>(), form<V, P, P, P, F, I, I, I, I, I, I, I, I, I, I, I>(), form<V, P, P, P, P, F, I, I, I, I, I, I, I, I, I, I, I>(),
      form<V, P, P, P, P, I, I, I, I, I, I, I, I, I, I, I, P, P, P, P, F, F>(), form<V, P, P, P, P, I, I, I, I, I, I, I, I, I, I, I, P, P, P, P, P, P, F, F, P, P, I>(),
      form<V, P, P, P, I, I, I, I, I, I, I, I, I>(), form<V, P, P, P, F, I, I, I, I, I, I, I, I, I>(), form<V, P, P, I, I, I, I, I, I, I, I>(),
      form<V, P, P, P, P, P, P, I, I, I, F>(), form<V, P, P, P, P, P, P, P, P, I, I, I, F, F>(), form<V, P, P, P, P, P, P, F, P, P, I, I, I>(),
      form<V, P, P, P, P, P, P, P, P, F, P, P, I, I, I>(), form<V, P, P, P, P, P, P, P, F, P, F, P, P, I, I, I>(),
      form<V, P, P, P, P, P, P, I, I, I, I>(), form<V, P, P, P, P, P, P, P, I, I, I>(), form<V, P, P, P, P, P, I, I, I, F, F>(),
      form<V, P, P, P, F, F, F, I, L>(), form<V, P, P, P, F, F, L>(), form<V, I, P, P, P, F>(), form<V, I, P, P, P, P, F, F, F, I>(),
  };
  for (const Form& f : forms)
    if (f.name == name) return f.invoke;
  return nullptr;
}

PyObject* call_vectorcall(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  Call* c = (Call*)self;
  if (PyVectorcall_NARGS(nargsf) == c->nargs && kwnames == nullptr) {
    bool ordinary = true;
    PyObject* r = c->invoke(c, args, ordinary);
    if (ordinary) return r;
  }
  return PyObject_Vectorcall(c->fallback, args, nargsf, kwnames);
}
void call_dealloc(PyObject* self) { Py_XDECREF(((Call*)self)->fallback); Py_TYPE(self)->tp_free(self); }
PyObject* call_getattro(PyObject* self, PyObject* name) {            // argtypes and the like: the ctypes function's
  PyObject* r = PyObject_GenericGetAttr(self, name);
  if (r || !PyErr_ExceptionMatches(PyExc_AttributeError)) return r;
  PyErr_Clear();
  return PyObject_GetAttr(((Call*)self)->fallback, name);
}
PyTypeObject CallType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// call(signature, address, ctypes function) -> callable, or the ctypes function itself where the signature is not one of the forms
PyObject* make_call(PyObject*, PyObject* args) {
  const char* name; unsigned long long address; PyObject* fallback;
  if (!PyArg_ParseTuple(args, "sKO", &name, &address, &fallback)) return nullptr;
  Invoke invoke = find_form(name);
  if (!invoke) { Py_INCREF(fallback); return fallback; }
  Call* c = PyObject_New(Call, &CallType);
  if (!c) return nullptr;
  Py_INCREF(fallback);
  c->vectorcall = call_vectorcall; c->fn = (void*)(uintptr_t)address; c->fallback = fallback; c->invoke = invoke; c->nargs = (Py_ssize_t)strlen(name) - 1;
  return (PyObject*)c;
}

// ---- check(): nothing while the byte at `flag` is 0, `raise_()` otherwise ----------------------------------------------------------
struct Check { PyObject_HEAD vectorcallfunc vectorcall; const volatile unsigned char* flag; PyObject* raise_; };
PyObject* check_vectorcall(PyObject* self, PyObject* const*, size_t nargsf, PyObject* kwnames) {
  Check* c = (Check*)self;
  if (PyVectorcall_NARGS(nargsf) != 0 || kwnames) { PyErr_SetString(PyExc_TypeError, "check() takes no arguments"); return nullptr; }
  if (*c->flag == 0) Py_RETURN_NONE;
  return PyObject_CallNoArgs(c->raise_);
}
void check_dealloc(PyObject* self) { Py_XDECREF(((Check*)self)->raise_); Py_TYPE(self)->tp_free(self); }
PyTypeObject CheckType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyObject* make_check(PyObject*, PyObject* args) {
  unsigned long long address; PyObject* raise_;
  if (!PyArg_ParseTuple(args, "KO", &address, &raise_)) return nullptr;
  Check* c = PyObject_New(Check, &CheckType);
  if (!c) return nullptr;
  Py_INCREF(raise_);
  c->vectorcall = check_vectorcall; c->flag = (const volatile unsigned char*)(uintptr_t)address; c->raise_ = raise_;
  return (PyObject*)c;
}

// ---- Buf: a span of backend memory (address, number of 4-byte elements, an owner to keep alive).  The collector follows it only where
// there is an owner (which may hold the Buf in turn): such a one is an OwnedBuf, the same for the caller.
struct Buf { PyObject_HEAD PyObject *ptr, *n, *keep; };
PyTypeObject BufType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject OwnedBufType = {PyVarObject_HEAD_INIT(nullptr, 0)};
inline PyObject* as_int(PyObject* o) {
  if (PyLong_CheckExact(o)) { Py_INCREF(o); return o; }
  return PyNumber_Long(o);
}
PyObject* buf_of(PyTypeObject* type, PyObject* ptr, PyObject* n, PyObject* keep) {           // takes over ptr and n
  if (type == &BufType && keep != Py_None) type = &OwnedBufType;
  Buf* b = ptr && n ? (Buf*)type->tp_alloc(type, 0) : nullptr;
  if (!b) { Py_XDECREF(ptr); Py_XDECREF(n); return nullptr; }
  Py_INCREF(keep);
  b->ptr = ptr; b->n = n; b->keep = keep;
  return (PyObject*)b;
}
PyObject* buf_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  static const char* names[] = {"ptr", "n", "keep", nullptr};
  PyObject *ptr, *n, *keep = Py_None;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "OO|O", (char**)names, &ptr, &n, &keep)) return nullptr;
  PyObject* p = as_int(ptr);
  return buf_of(type, p, p ? as_int(n) : nullptr, keep);
}
PyObject* buf_vectorcall(PyObject* type, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  const Py_ssize_t nargs = PyVectorcall_NARGS(nargsf);
  if ((nargs == 2 || nargs == 3) && !kwnames) {
    PyObject* p = as_int(args[0]);
    return buf_of((PyTypeObject*)type, p, p ? as_int(args[1]) : nullptr, nargs == 3 ? args[2] : Py_None);
  }
  PyObject* t = PyTuple_New(nargs);
  if (!t) return nullptr;
  for (Py_ssize_t i = 0; i < nargs; i++) { Py_INCREF(args[i]); PyTuple_SET_ITEM(t, i, args[i]); }
  PyObject* kw = kwnames ? PyDict_New() : nullptr;
  for (Py_ssize_t i = 0; kwnames && kw && i < PyTuple_GET_SIZE(kwnames); i++) PyDict_SetItem(kw, PyTuple_GET_ITEM(kwnames, i), args[nargs + i]);
  PyObject* r = buf_new((PyTypeObject*)type, t, kw);
  Py_DECREF(t); Py_XDECREF(kw);
  return r;
}
void buf_dealloc(PyObject* self) {
  Buf* b = (Buf*)self;
  Py_XDECREF(b->ptr); Py_XDECREF(b->n); Py_XDECREF(b->keep);
  Py_TYPE(self)->tp_free(self);
}
void owned_buf_dealloc(PyObject* self) { PyObject_GC_UnTrack(self); buf_dealloc(self); }
int buf_traverse(PyObject* self, visitproc visit, void* arg) { Buf* b = (Buf*)self; Py_VISIT(b->ptr); Py_VISIT(b->n); Py_VISIT(b->keep); return 0; }
int buf_clear(PyObject* self) { Buf* b = (Buf*)self; Py_CLEAR(b->keep); return 0; }
// offset(k, n=None): the same memory, starting k elements in
PyObject* buf_offset(PyObject* self, PyObject* args, PyObject* kw) {
  static const char* names[] = {"k", "n", nullptr};
  Buf* b = (Buf*)self;
  PyObject *k, *n = Py_None;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "O|O", (char**)names, &k, &n)) return nullptr;
  if (!b->ptr || !b->n || !b->keep) { PyErr_SetString(PyExc_AttributeError, "ptr"); return nullptr; }
  PyObject* i = PyNumber_Long(k);
  PyObject* four = i ? PyLong_FromLong(4) : nullptr;
  PyObject* bytes = four ? PyNumber_Multiply(four, i) : nullptr;
  PyObject* p = bytes ? PyNumber_Add(b->ptr, bytes) : nullptr;
  PyObject* left = !p ? nullptr : n == Py_None ? PyNumber_Subtract(b->n, i) : as_int(n);
  PyObject* r = buf_of(&BufType, p, left, b->keep);
  Py_XDECREF(i); Py_XDECREF(four); Py_XDECREF(bytes);
  return r;
}
PyObject* buf_reduce(PyObject* self, PyObject*) { Buf* b = (Buf*)self; return Py_BuildValue("O(OOO)", (PyObject*)&BufType, b->ptr, b->n, b->keep); }
PyMemberDef buf_members[] = {{"ptr", T_OBJECT_EX, offsetof(Buf, ptr), 0, nullptr}, {"n", T_OBJECT_EX, offsetof(Buf, n), 0, nullptr}, {"keep", T_OBJECT_EX, offsetof(Buf, keep), 0, nullptr}, {}};
PyMethodDef buf_methods[] = {{"offset", (PyCFunction)(void (*)(void))buf_offset, METH_VARARGS | METH_KEYWORDS, "The same memory, starting k elements in."},
                             {"__reduce__", buf_reduce, METH_NOARGS, nullptr}, {}};

PyMethodDef methods[] = {{"call", make_call, METH_VARARGS, nullptr}, {"check", make_check, METH_VARARGS, nullptr}, {}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_lhpy", nullptr, -1, methods};
}  // namespace

PyMODINIT_FUNC PyInit__lhpy(void) {
  PyObject* ctypes = PyImport_ImportModule("ctypes");
  if (!ctypes) return nullptr;
  g_array_type = PyObject_GetAttrString(ctypes, "Array");
  Py_DECREF(ctypes);
  if (!g_array_type) return nullptr;
  CallType.tp_name = "lantern_amd._lhpy.Call"; CallType.tp_basicsize = sizeof(Call); CallType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  CallType.tp_vectorcall_offset = offsetof(Call, vectorcall); CallType.tp_call = PyVectorcall_Call; CallType.tp_dealloc = call_dealloc; CallType.tp_getattro = call_getattro;
  CheckType.tp_name = "lantern_amd._lhpy.Check"; CheckType.tp_basicsize = sizeof(Check); CheckType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  CheckType.tp_vectorcall_offset = offsetof(Check, vectorcall); CheckType.tp_call = PyVectorcall_Call; CheckType.tp_dealloc = check_dealloc;
  BufType.tp_name = "lantern_amd.backend.Buf"; BufType.tp_basicsize = sizeof(Buf); BufType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
  BufType.tp_doc = "A span of backend memory: address, element count (4-byte elements) and an owner to keep alive.";
  BufType.tp_new = buf_new; BufType.tp_vectorcall = buf_vectorcall; BufType.tp_dealloc = buf_dealloc; BufType.tp_members = buf_members; BufType.tp_methods = buf_methods;
  BufType.tp_traverse = buf_traverse; BufType.tp_clear = buf_clear;           // (for classes derived from it, which the collector follows)
  OwnedBufType.tp_name = BufType.tp_name; OwnedBufType.tp_basicsize = sizeof(Buf); OwnedBufType.tp_base = &BufType; OwnedBufType.tp_doc = BufType.tp_doc;
  OwnedBufType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
  OwnedBufType.tp_dealloc = owned_buf_dealloc; OwnedBufType.tp_traverse = buf_traverse; OwnedBufType.tp_clear = buf_clear; OwnedBufType.tp_free = PyObject_GC_Del;
  if (PyType_Ready(&CallType) < 0 || PyType_Ready(&CheckType) < 0 || PyType_Ready(&BufType) < 0 || PyType_Ready(&OwnedBufType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&BufType);
  if (PyModule_AddObject(m, "Buf", (PyObject*)&BufType) < 0) { Py_DECREF(&BufType); Py_DECREF(m); return nullptr; }
  return m;
}
