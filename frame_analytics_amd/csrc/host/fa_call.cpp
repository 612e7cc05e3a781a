// Calls into libfa_gpu.so from Python without ctypes' marshalling.
//
// A scoring call of one small frame is host time: ctypes converts the 17 to 27
// arguments of an entry point through its argtypes objects, ~2.5 us a call of
// the ~12 us that fa.psnr on a 512 x 512 frame takes.  Here each entry point's
// prototype (include/fa_abi.h) is taken apart at compile time, so an argument is
// one PyLong / PyFloat conversion.
//
// entry(name, address, prototype) returns a callable for the entry point `name` at
// `address` (where the caller's loaded library has it), or None unless the
// argument types compiled in here are `prototype`, one letter each (p pointer, i
// int, l int64, d double): a module older than the library never calls through
// another prototype.  Its arguments: integers, floats, None or
// an address for pointers, or a ctypes array for a
// host array.  A wrong count or type raises before the library is entered.  The
// GIL is released around the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstddef>
#include <cstdint>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "fa_abi.h"

namespace {

// Buffers borrowed for the time of one call (host arrays of strides, weights,
// pointers: at most a handful).
struct Borrowed {
  static constexpr int MAX = 8;
  Py_buffer b[MAX];
  int n = 0;
  ~Borrowed() {
    for (int i = 0; i < n; ++i) PyBuffer_Release(&b[i]);
  }
};

PyObject* array_type = nullptr;  // ctypes.Array

template <typename T>
bool convert(PyObject* o, T* out, Borrowed& held) {
  if constexpr (std::is_pointer<T>::value) {
    if (o == Py_None) {
      *out = nullptr;
      return true;
    }
    if (PyLong_Check(o)) {
      void* p = PyLong_AsVoidPtr(o);
      if (!p && PyErr_Occurred()) return false;
      *out = reinterpret_cast<T>(p);
      return true;
    }
    // ctypes arrays alone: another object with a buffer may stand for an address
    // (a ctypes.c_void_p is one, whose buffer holds it), which ctypes resolves
    const int is_array = PyObject_IsInstance(o, array_type);
    if (is_array <= 0) {
      if (is_array == 0)
        PyErr_Format(PyExc_TypeError, "no address or ctypes array: %.80s", Py_TYPE(o)->tp_name);
      return false;
    }
    if (held.n == Borrowed::MAX) {
      PyErr_SetString(PyExc_TypeError, "too many array arguments");
      return false;
    }
    if (PyObject_GetBuffer(o, &held.b[held.n], PyBUF_SIMPLE) != 0) return false;
    *out = reinterpret_cast<T>(held.b[held.n].buf);
    ++held.n;
    return true;
  } else if constexpr (std::is_floating_point<T>::value) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) return false;
    *out = static_cast<T>(v);
    return true;
  } else {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) return false;
    *out = static_cast<T>(v);  // as ctypes: the low bits
    return true;
  }
}

template <typename... A, std::size_t... I>
PyObject* invoke(int (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
  std::tuple<A...> v{};
  Borrowed held;
  if (!(convert(args[I], &std::get<I>(v), held) && ...)) return nullptr;
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS;
  rc = fn(std::get<I>(v)...);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(rc);
}

struct Entry {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  void* address;
  const char* name;
};

template <typename... A>
PyObject* call(int (*)(A...), PyObject* self, PyObject* const* args, size_t nargsf,
               PyObject* kwnames) {
  const Entry* e = reinterpret_cast<Entry*>(self);
  if (kwnames && PyTuple_GET_SIZE(kwnames) > 0) {
    PyErr_Format(PyExc_TypeError, "%s takes no keyword arguments", e->name);
    return nullptr;
  }
  if (PyVectorcall_NARGS(nargsf) != static_cast<Py_ssize_t>(sizeof...(A))) {
    PyErr_Format(PyExc_TypeError, "%s takes %zu arguments (%zd given)", e->name, sizeof...(A),
                 PyVectorcall_NARGS(nargsf));
    return nullptr;
  }
  return invoke(reinterpret_cast<int (*)(A...)>(e->address), args,
                std::index_sequence_for<A...>{});
}

template <typename T>
constexpr char letter() {
  if constexpr (std::is_pointer<T>::value) return 'p';
  else if constexpr (std::is_same<T, double>::value) return 'd';
  else if constexpr (std::is_same<T, int>::value) return 'i';
  else if constexpr (std::is_same<T, int64_t>::value) return 'l';
  else return '!';  // none that Python can name
}

template <typename... A>
const char* prototype(int (*)(A...)) {
  static const char s[] = {letter<A>()..., '\0'};
  return s;
}

#define FA_ENTRY(NAME)                                                                   \
  {#NAME, prototype(decltype(&NAME)(nullptr)), [](PyObject* self, PyObject* const* args, size_t n, PyObject* kw) -> PyObject* { \
     return call(decltype(&NAME)(nullptr), self, args, n, kw);                           \
   }}

struct Known {
  const char* name;
  const char* types;
  vectorcallfunc fn;
};

const Known KNOWN[] = {
    FA_ENTRY(fa_gpu_pixel_reduce_once), FA_ENTRY(fa_gpu_pixel_reduce_ex),
    FA_ENTRY(fa_gpu_ssim),              FA_ENTRY(fa_gpu_ssim_ex),
    FA_ENTRY(fa_gpu_ssim_once),         FA_ENTRY(fa_gpu_ssim_cs),
    FA_ENTRY(fa_gpu_ssim_cs_coef),      FA_ENTRY(fa_gpu_ssim_cs_scatter),
    FA_ENTRY(fa_gpu_ssim_backward),
    FA_ENTRY(fa_gpu_ms_ssim),           FA_ENTRY(fa_gpu_ms_ssim_head),
    FA_ENTRY(fa_gpu_ms_ssim_head_backward), FA_ENTRY(fa_gpu_gmsd_ex),
    FA_ENTRY(fa_gpu_gmsd_once),         FA_ENTRY(fa_gpu_gmsd_backward),
};

void entry_dealloc(PyObject* self) { Py_TYPE(self)->tp_free(self); }

PyTypeObject entry_type = [] {
  PyTypeObject t = {PyVarObject_HEAD_INIT(nullptr, 0)};
  t.tp_name = "_fa_call.Entry";
  t.tp_basicsize = sizeof(Entry);
  t.tp_dealloc = entry_dealloc;
  t.tp_vectorcall_offset = offsetof(Entry, vectorcall);
  t.tp_call = PyVectorcall_Call;
  t.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  return t;
}();

PyObject* make_entry(PyObject*, PyObject* args) {
  const char* name = nullptr;
  PyObject* address = nullptr;
  const char* types = nullptr;
  if (!PyArg_ParseTuple(args, "sOs", &name, &address, &types)) return nullptr;
  void* p = PyLong_AsVoidPtr(address);
  if (!p) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
    return nullptr;
  }
  for (const Known& k : KNOWN) {
    if (std::strcmp(k.name, name) != 0 || std::strcmp(k.types, types) != 0) continue;
    Entry* e = PyObject_New(Entry, &entry_type);
    if (!e) return nullptr;
    e->vectorcall = k.fn;
    e->address = p;
    e->name = k.name;
    return reinterpret_cast<PyObject*>(e);
  }
  Py_RETURN_NONE;  // not one of the calls that run often, or another: ctypes serves it
}

PyMethodDef methods[] = {
    {"entry", make_entry, METH_VARARGS, "entry(name, address, prototype) -> callable, or None"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fa_call", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fa_call() {
  if (PyType_Ready(&entry_type) < 0) return nullptr;
  PyObject* ctypes = PyImport_ImportModule("ctypes");
  if (!ctypes) return nullptr;
  array_type = PyObject_GetAttrString(ctypes, "Array");
  Py_DECREF(ctypes);
  if (!array_type) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddIntConstant(m, "abi_version", FA_ABI_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
