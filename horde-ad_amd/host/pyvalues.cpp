// The values of hostapi.py and their calls into libhordead_host.so as a CPython extension.
//
// A program over the carrier is some hundred calls of a few hundred nanoseconds each.  Through ctypes a call costs 2 to 3 us more:
// arguments converted one by one, a list made into a C array element by element, an output cell, a Python object with a
// finalizer that is again such a call.  Here a value is a C object (its handle goes back in its deallocator), and a `Fn`
// is an entry point with a signature that says how its arguments are laid out:
//
//   v  a value          x  a lane value        i  an int             n  an int64_t       d  a double         p  an address (an int)
//   S  sizes, as their number and an int64_t array (whatever int() takes)         Q  ints, as their number and an int array
//   K  lane values, as their number and an array of handles
//
// after the host, whose context handle is the first argument of every call.  What comes back: "V" a value, "X" a lane value
// (over the index space of the S argument, or of the first lane value among the arguments, or of the value), "N" nothing.
// Calls release the interpreter's lock, as ctypes' do.  The entry points' addresses come from Python, which has the library
// loaded (a test may load another build of it).
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <climits>
#include <cstdint>
#include <cstring>

namespace {

struct HostBase { PyObject_HEAD void* ctx; };
struct Val { PyObject_HEAD PyObject* host; void* h; };
struct Lane { PyObject_HEAD PyObject* host; void* h; PyObject* shm; };

PyTypeObject *value_type, *lane_type;      // the classes of hostapi.py that stand on these
PyObject* error_type;
int (*p_free)(void*);
int (*p_ix_free)(void*);
int (*p_rank)(void*);
int (*p_dtype)(void*);
int (*p_shape)(void*, int64_t*);
int (*p_ix_dtype)(void*);
const char* (*p_last_error)(void*);
int (*p_backward)(void*, void*, void*, int, void**, void**);

constexpr int kMaxRank = 64;

extern PyTypeObject HostBaseType, ValType, LaneType, FnType;

// An address as Python hands it over: an int, None, or a ctypes pointer.
bool address(PyObject* o, void** out) {
  if (o == Py_None) { *out = nullptr; return true; }
  if (PyLong_Check(o)) {
    *out = PyLong_AsVoidPtr(o);
    return !PyErr_Occurred();
  }
  PyObject* v = PyObject_GetAttrString(o, "value");
  if (!v) return false;
  const bool ok = v == Py_None ? (*out = nullptr, true) : PyLong_Check(v) ? (*out = PyLong_AsVoidPtr(v), !PyErr_Occurred()) : (PyErr_SetString(PyExc_TypeError, "not an address"), false);
  Py_DECREF(v);
  return ok;
}

PyObject* raise_status(void* ctx, int rc) {
  PyObject* e = PyObject_CallFunction(error_type, "is", rc, p_last_error(ctx));
  if (e) {
    PyErr_SetObject(error_type, e);
    Py_DECREF(e);
  }
  return nullptr;
}

// ---- the host ------------------------------------------------------------
PyObject* host_bind(PyObject* self, PyObject* h) {
  if (!address(h, &((HostBase*)self)->ctx)) return nullptr;
  Py_RETURN_NONE;
}
void host_dealloc(PyObject* self) { Py_TYPE(self)->tp_free(self); }
PyMethodDef host_methods[] = {{"_bind", host_bind, METH_O, "the context's handle"}, {nullptr, nullptr, 0, nullptr}};

// ---- values --------------------------------------------------------------
PyObject* make_value(PyObject* host, void* h) {
  Val* v = (Val*)value_type->tp_alloc(value_type, 0);
  if (!v) { p_free(h); return nullptr; }
  Py_INCREF(host);
  v->host = host;
  v->h = h;
  return (PyObject*)v;
}
int val_init(PyObject* self, PyObject* args, PyObject* kw) {
  PyObject *host, *h;
  static const char* names[] = {"host", "h", nullptr};
  if (!PyArg_ParseTupleAndKeywords(args, kw, "OO", (char**)names, &host, &h)) return -1;
  Val* v = (Val*)self;
  void* p;
  if (!address(h, &p)) return -1;
  if (v->h) p_free(v->h);
  v->h = p;
  Py_INCREF(host);
  Py_XSETREF(v->host, host);
  return 0;
}
int val_traverse(PyObject* self, visitproc visit, void* arg) {
  Py_VISIT(((Val*)self)->host);
  return 0;
}
int val_clear(PyObject* self) {
  Py_CLEAR(((Val*)self)->host);
  return 0;
}
void val_dealloc(PyObject* self) {
  PyObject_GC_UnTrack(self);
  Val* v = (Val*)self;
  if (v->h) p_free(v->h);
  v->h = nullptr;
  val_clear(self);
  Py_TYPE(self)->tp_free(self);
}
PyObject* val_h(PyObject* self, void*) {
  if (!((Val*)self)->h) Py_RETURN_NONE;
  return PyLong_FromVoidPtr(((Val*)self)->h);
}
PyObject* shape_tuple(void* h) {
  int64_t s[kMaxRank];
  const int r = p_rank(h);
  if (r < 0 || r > kMaxRank) { PyErr_SetString(PyExc_ValueError, "rank"); return nullptr; }
  p_shape(h, s);
  PyObject* t = PyTuple_New(r);
  for (int i = 0; t && i < r; ++i) {
    PyObject* e = PyLong_FromLongLong(s[i]);
    if (!e) { Py_CLEAR(t); break; }
    PyTuple_SET_ITEM(t, i, e);
  }
  return t;
}
PyObject* val_shape(PyObject* self, void*) { return shape_tuple(((Val*)self)->h); }
PyObject* val_dtype(PyObject* self, void*) { return PyLong_FromLong(p_dtype(((Val*)self)->h)); }
PyMemberDef val_members[] = {{"host", T_OBJECT_EX, offsetof(Val, host), READONLY, nullptr}, {nullptr, 0, 0, 0, nullptr}};
PyGetSetDef val_getset[] = {{"h", val_h, nullptr, "the handle", nullptr}, {"shape", val_shape, nullptr, nullptr, nullptr}, {"dtype", val_dtype, nullptr, nullptr, nullptr},
                            {nullptr, nullptr, nullptr, nullptr, nullptr}};

// ---- lane values ---------------------------------------------------------
PyObject* make_lane(PyObject* host, void* h, PyObject* shm) {
  Lane* v = (Lane*)lane_type->tp_alloc(lane_type, 0);
  if (!v) { p_ix_free(h); return nullptr; }
  Py_INCREF(host);
  Py_INCREF(shm);
  v->host = host;
  v->h = h;
  v->shm = shm;
  return (PyObject*)v;
}
int lane_init(PyObject* self, PyObject* args, PyObject* kw) {
  PyObject *host, *h, *shm;
  static const char* names[] = {"host", "h", "shm", nullptr};
  if (!PyArg_ParseTupleAndKeywords(args, kw, "OOO", (char**)names, &host, &h, &shm)) return -1;
  Lane* v = (Lane*)self;
  void* p;
  if (!address(h, &p)) return -1;
  if (v->h) p_ix_free(v->h);
  v->h = p;
  Py_INCREF(host);
  Py_XSETREF(v->host, host);
  Py_INCREF(shm);
  Py_XSETREF(v->shm, shm);
  return 0;
}
int lane_traverse(PyObject* self, visitproc visit, void* arg) {
  Py_VISIT(((Lane*)self)->host);
  Py_VISIT(((Lane*)self)->shm);
  return 0;
}
int lane_clear(PyObject* self) {
  Py_CLEAR(((Lane*)self)->host);
  Py_CLEAR(((Lane*)self)->shm);
  return 0;
}
void lane_dealloc(PyObject* self) {
  PyObject_GC_UnTrack(self);
  Lane* v = (Lane*)self;
  if (v->h) p_ix_free(v->h);
  v->h = nullptr;
  lane_clear(self);
  Py_TYPE(self)->tp_free(self);
}
PyObject* lane_h(PyObject* self, void*) {
  if (!((Lane*)self)->h) Py_RETURN_NONE;
  return PyLong_FromVoidPtr(((Lane*)self)->h);
}
PyObject* lane_dtype(PyObject* self, void*) { return PyLong_FromLong(p_ix_dtype(((Lane*)self)->h)); }
PyMemberDef lane_members[] = {{"host", T_OBJECT_EX, offsetof(Lane, host), READONLY, nullptr}, {"shm", T_OBJECT_EX, offsetof(Lane, shm), READONLY, nullptr}, {nullptr, 0, 0, 0, nullptr}};
PyGetSetDef lane_getset[] = {{"h", lane_h, nullptr, "the handle", nullptr}, {"dtype", lane_dtype, nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr, nullptr, nullptr}};

// ---- calls ---------------------------------------------------------------
// Integers and addresses are handed over in the integer registers and, from the seventh on, on the stack, a double in the first
// vector register wherever it stands among the parameters (System V, x86-64): one prototype fits every entry point.
typedef int (*Call)(int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, double);
struct Fn {
  PyObject_HEAD
  vectorcallfunc call;
  Call entry;
  char sig[12];
  char out;
};

// What stands for an integer (numpy's integers too, no fractions and no texts), from lo to hi
bool integer(PyObject* o, int64_t* out, int64_t lo, int64_t hi) {
  PyObject* l = PyNumber_Index(o);
  if (!l) return false;
  *out = PyLong_AsLongLong(l);
  Py_DECREF(l);
  if (*out == -1 && PyErr_Occurred()) return false;
  if (*out >= lo && *out <= hi) return true;
  PyErr_SetString(PyExc_OverflowError, "an integer is too large for its parameter");
  return false;
}
bool integer(PyObject* o, int64_t* out) { return integer(o, out, INT64_MIN, INT64_MAX); }
bool small_integer(PyObject* o, int64_t* out) { return integer(o, out, INT_MIN, INT_MAX); }
// One of a list of sizes: int() of it
bool size(PyObject* o, int64_t* out) {
  if (PyLong_Check(o)) return integer(o, out);
  PyObject* l = PyNumber_Long(o);
  const bool ok = l && integer(l, out);
  Py_XDECREF(l);
  return ok;
}

PyObject* fn_call(PyObject* self, PyObject* const* args, size_t nf, PyObject* kw) {
  const Fn* f = (const Fn*)self;
  const Py_ssize_t n = PyVectorcall_NARGS(nf);
  if ((kw && PyTuple_GET_SIZE(kw)) || n != 1 + (Py_ssize_t)strlen(f->sig)) { PyErr_Format(PyExc_TypeError, "expected the host and %d arguments", (int)strlen(f->sig)); return nullptr; }
  if (!PyObject_TypeCheck(args[0], &HostBaseType)) { PyErr_SetString(PyExc_TypeError, "not a host"); return nullptr; }
  void* ctx = ((HostBase*)args[0])->ctx;
  int64_t a[8] = {(int64_t)ctx, 0, 0, 0, 0, 0, 0, 0};
  int na = 1;
  double d = 0;
  int64_t lists[2][kMaxRank];
  int n_lists = 0;
  PyObject *space = nullptr, *seq = nullptr, *lanes = nullptr;      // the index space of a lane value, a sequence at hand, the lane values of a K argument
  const Val* first = nullptr;
  auto stop = [&]() -> PyObject* {
    Py_XDECREF(seq);
    Py_XDECREF(lanes);
    Py_XDECREF(space);
    return nullptr;
  };
  auto over = [&](const PyObject* lane) {
    if (space) return;
    space = ((const Lane*)lane)->shm;
    Py_XINCREF(space);
  };
  for (int k = 0; f->sig[k]; ++k) {
    PyObject* o = args[k + 1];
    const char c = f->sig[k];
    if (c == 'v') {
      if (!PyObject_TypeCheck(o, &ValType)) { PyErr_Format(PyExc_TypeError, "argument %d is not a value", k + 1); return stop(); }
      if (!first) first = (Val*)o;
      a[na++] = (int64_t)((Val*)o)->h;
    } else if (c == 'x') {
      if (!PyObject_TypeCheck(o, &LaneType)) { PyErr_Format(PyExc_TypeError, "argument %d is not a lane value", k + 1); return stop(); }
      over(o);
      a[na++] = (int64_t)((Lane*)o)->h;
    } else if (c == 'i') {
      if (!small_integer(o, &a[na++])) return stop();
    } else if (c == 'n') {
      if (!integer(o, &a[na++])) return stop();
    } else if (c == 'p') {
      if (!address(o, (void**)&a[na++])) return stop();
    } else if (c == 'd') {
      d = PyFloat_AsDouble(o);
      if (d == -1 && PyErr_Occurred()) return stop();
    } else {      // S, Q, K
      // (lane values are kept by a tuple until the call is over: an iterator's are nobody else's, and a list may change while other threads run)
      seq = c == 'K' ? PySequence_Tuple(o) : PySequence_Fast(o, "a sequence is expected");
      if (!seq) return stop();
      const Py_ssize_t len = PySequence_Fast_GET_SIZE(seq);
      if (len > kMaxRank) { PyErr_SetString(PyExc_ValueError, "too many dims"); return stop(); }
      int64_t* l = lists[n_lists++];
      for (Py_ssize_t i = 0; i < len; ++i) {
        PyObject* e = PySequence_Fast_GET_ITEM(seq, i);
        if (c == 'K') {
          if (!PyObject_TypeCheck(e, &LaneType)) { PyErr_Format(PyExc_TypeError, "index %d is not a lane value", (int)i); return stop(); }
          over(e);
          l[i] = (int64_t)((Lane*)e)->h;
        } else {
          int64_t v;
          if (!(c == 'Q' ? small_integer(e, &v) : size(e, &v))) return stop();
          if (c == 'Q') ((int*)l)[i] = (int)v;
          else l[i] = v;
        }
      }
      a[na++] = (int64_t)len;
      a[na++] = (int64_t)l;
      if (c == 'S' && f->out == 'X') {
        Py_XSETREF(space, PyTuple_New(len));
        for (Py_ssize_t i = 0; space && i < len; ++i) {
          PyObject* e = PyLong_FromLongLong(l[i]);
          if (!e) return stop();
          PyTuple_SET_ITEM(space, i, e);
        }
        if (!space) return stop();
      }
      if (c == 'K') lanes = seq, seq = nullptr;
      else Py_CLEAR(seq);
    }
  }
  void* out = nullptr;
  if (f->out != 'N') a[na++] = (int64_t)&out;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f->entry(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], d);
  Py_END_ALLOW_THREADS
  if (rc) {
    stop();
    return raise_status(ctx, rc);
  }
  if (f->out == 'X' && !space && first) space = shape_tuple(first->h);
  PyObject* r = nullptr;
  if (f->out == 'V') {
    r = make_value(args[0], out);
  } else if (f->out == 'N') {
    r = Py_None;
    Py_INCREF(r);
  } else if (space) {
    r = make_lane(args[0], out, space);
  } else {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "no index space");
    p_ix_free(out);
  }
  stop();
  return r;
}

PyObject* fn_new(PyTypeObject* type, PyObject* args, PyObject*) {
  PyObject* at;
  const char *sig, *out;
  if (!PyArg_ParseTuple(args, "Oss", &at, &sig, &out)) return nullptr;
  int words = 1 + (out[0] != 'N'), lists = 0, doubles = 0, kept = 0;
  for (const char* c = sig; *c; ++c) {
    if (!strchr("vxindpSQK", *c)) { PyErr_SetString(PyExc_ValueError, "unknown letter in a signature"); return nullptr; }
    const bool list = *c == 'S' || *c == 'Q' || *c == 'K';
    words += list ? 2 : *c != 'd';
    lists += list;
    doubles += *c == 'd';
    kept += *c == 'K';
  }
  if (strlen(sig) >= sizeof(Fn::sig) || words > 8 || lists > 2 || doubles > 1 || kept > 1 || !strchr("VXN", out[0])) { PyErr_SetString(PyExc_ValueError, "signature"); return nullptr; }
  void* p;
  if (!address(at, &p)) return nullptr;
  Fn* f = (Fn*)type->tp_alloc(type, 0);
  if (!f) return nullptr;
  f->call = fn_call;
  f->entry = (Call)p;
  strcpy(f->sig, sig);
  f->out = out[0];
  return (PyObject*)f;
}
void fn_dealloc(PyObject* self) { Py_TYPE(self)->tp_free(self); }

PyObject* backward(PyObject*, PyObject* args) {      // host, out, dt or None, inputs
  PyObject *host, *out, *dt, *inputs;
  if (!PyArg_ParseTuple(args, "O!O!OO", &HostBaseType, &host, &ValType, &out, &dt, &inputs)) return nullptr;
  if (dt != Py_None && !PyObject_TypeCheck(dt, &ValType)) { PyErr_SetString(PyExc_TypeError, "the cotangent is not a value"); return nullptr; }
  PyObject* seq = PySequence_Tuple(inputs);      // (keeps the values until the call is over)
  if (!seq) return nullptr;
  const Py_ssize_t n = PyTuple_GET_SIZE(seq);
  void** h = (void**)PyMem_Calloc((size_t)(n ? 2 * n : 1), sizeof(void*));
  if (!h) { Py_DECREF(seq); return PyErr_NoMemory(); }
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* e = PyTuple_GET_ITEM(seq, i);
    if (!PyObject_TypeCheck(e, &ValType)) {
      PyErr_Format(PyExc_TypeError, "input %d is not a value", (int)i);
      PyMem_Free(h);
      Py_DECREF(seq);
      return nullptr;
    }
    h[i] = ((Val*)e)->h;
  }
  void* ctx = ((HostBase*)host)->ctx;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = p_backward(ctx, ((Val*)out)->h, dt == Py_None ? nullptr : ((Val*)dt)->h, (int)n, h, h + n);
  Py_END_ALLOW_THREADS
  PyObject* r = nullptr;
  if (rc) {
    raise_status(ctx, rc);
  } else if ((r = PyList_New(n))) {
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* v = r ? make_value(host, h[n + i]) : (p_free(h[n + i]), nullptr);
      if (!v) Py_CLEAR(r);
      else PyList_SET_ITEM(r, i, v);
    }
  } else {
    for (Py_ssize_t i = 0; i < n; ++i) p_free(h[n + i]);
  }
  PyMem_Free(h);
  Py_DECREF(seq);
  return r;
}

PyObject* setup(PyObject*, PyObject* args) {      // the classes, the error, and the addresses of what values need
  PyObject *v, *x, *e, *at[8];
  if (!PyArg_ParseTuple(args, "O!O!OOOOOOOOO", &PyType_Type, &v, &PyType_Type, &x, &e, &at[0], &at[1], &at[2], &at[3], &at[4], &at[5], &at[6], &at[7])) return nullptr;
  if (!PyType_IsSubtype((PyTypeObject*)v, &ValType) || !PyType_IsSubtype((PyTypeObject*)x, &LaneType)) { PyErr_SetString(PyExc_TypeError, "classes"); return nullptr; }
  void* p[8];
  for (int i = 0; i < 8; ++i)
    if (!address(at[i], &p[i])) return nullptr;
  Py_INCREF(v);
  Py_INCREF(x);
  Py_INCREF(e);
  value_type = (PyTypeObject*)v;
  lane_type = (PyTypeObject*)x;
  error_type = e;
  memcpy(&p_free, &p[0], sizeof p[0]);
  memcpy(&p_ix_free, &p[1], sizeof p[0]);
  memcpy(&p_rank, &p[2], sizeof p[0]);
  memcpy(&p_dtype, &p[3], sizeof p[0]);
  memcpy(&p_shape, &p[4], sizeof p[0]);
  memcpy(&p_ix_dtype, &p[5], sizeof p[0]);
  memcpy(&p_last_error, &p[6], sizeof p[0]);
  memcpy(&p_backward, &p[7], sizeof p[0]);
  Py_RETURN_NONE;
}

PyTypeObject HostBaseType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject ValType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject LaneType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject FnType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyMethodDef functions[] = {{"backward", backward, METH_VARARGS, "cotangents of the inputs"}, {"setup", setup, METH_VARARGS, "classes and entry points"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pyvalues", "values of the host layer", -1, functions, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pyvalues() {
  HostBaseType.tp_name = "_pyvalues.HostBase";
  HostBaseType.tp_basicsize = sizeof(HostBase);
  HostBaseType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
  HostBaseType.tp_new = PyType_GenericNew;
  HostBaseType.tp_dealloc = host_dealloc;
  HostBaseType.tp_methods = host_methods;
  ValType.tp_name = "_pyvalues.Val";
  ValType.tp_basicsize = sizeof(Val);
  ValType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
  ValType.tp_new = PyType_GenericNew;
  ValType.tp_init = val_init;
  ValType.tp_dealloc = val_dealloc;
  ValType.tp_traverse = val_traverse;
  ValType.tp_clear = val_clear;
  ValType.tp_members = val_members;
  ValType.tp_getset = val_getset;
  LaneType.tp_name = "_pyvalues.Lane";
  LaneType.tp_basicsize = sizeof(Lane);
  LaneType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
  LaneType.tp_new = PyType_GenericNew;
  LaneType.tp_init = lane_init;
  LaneType.tp_dealloc = lane_dealloc;
  LaneType.tp_traverse = lane_traverse;
  LaneType.tp_clear = lane_clear;
  LaneType.tp_members = lane_members;
  LaneType.tp_getset = lane_getset;
  FnType.tp_name = "_pyvalues.Fn";
  FnType.tp_basicsize = sizeof(Fn);
  FnType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  FnType.tp_new = fn_new;
  FnType.tp_dealloc = fn_dealloc;
  FnType.tp_call = PyVectorcall_Call;
  FnType.tp_vectorcall_offset = offsetof(Fn, call);
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  if (PyModule_AddStringConstant(m, "SOURCE", PYVALUES_SOURCE) < 0) { Py_DECREF(m); return nullptr; }
  struct { const char* name; PyTypeObject* t; } types[] = {{"HostBase", &HostBaseType}, {"Val", &ValType}, {"Lane", &LaneType}, {"Fn", &FnType}};
  for (auto& t : types) {
    if (PyType_Ready(t.t) < 0) { Py_DECREF(m); return nullptr; }
    Py_INCREF(t.t);
    if (PyModule_AddObject(m, t.name, (PyObject*)t.t) < 0) { Py_DECREF(t.t); Py_DECREF(m); return nullptr; }
  }
  return m;
}
