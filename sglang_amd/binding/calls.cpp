// Python calls of the C ABI without ctypes, which takes 0.09 us an argument (3.1 us for the 34 of an extend attention with its store, 0.27 here; a
// forward_extend of 37 cold tokens, 14 / 2 heads, 22.0 -> 20.7 us).  The header's own types say how an argument is converted; the names come from the same header
// (build.py).  A value that is neither a whole number, a float nor None (a ctypes object) makes a call return NotImplemented: native.call() then goes the long way.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>

#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "sglang_amd.h"

namespace {

// what ctypes takes for c_void_p, c_int64 / c_int (which cut a value to their width as it does) and c_float
template <typename T>
bool take(PyObject* o, T& v) {
  if constexpr (std::is_pointer_v<T>) {
    if (o != Py_None && !PyLong_Check(o)) return false;
    v = o == Py_None ? nullptr : reinterpret_cast<T>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
  } else if constexpr (std::is_floating_point_v<T>) {
    const double d = PyFloat_Check(o) ? PyFloat_AS_DOUBLE(o) : PyLong_Check(o) ? PyLong_AsDouble(o) : -1.0;
    if (!PyFloat_Check(o) && (!PyLong_Check(o) || (d == -1.0 && PyErr_Occurred()))) {
      PyErr_Clear();
      return false;
    }
    v = static_cast<T>(d);
  } else {
    if (!PyLong_Check(o)) return false;
    v = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
  }
  return true;
}

template <typename R, typename... A, size_t... I>
PyObject* invoke(R (*fn)(A...), PyObject* const* a, std::index_sequence<I...>) {
  std::tuple<std::remove_const_t<A>...> v;
  if (!(take(a[I], std::get<I>(v)) && ...)) Py_RETURN_NOTIMPLEMENTED;
  R r;
  Py_BEGIN_ALLOW_THREADS
  r = fn(std::get<I>(v)...);
  Py_END_ALLOW_THREADS
  return PyLong_FromLongLong(static_cast<long long>(r));
}

// NUMBER: the function's place in SGL_AMD_NAMES
template <int NUMBER, typename F>
struct Call;
template <int NUMBER, typename R, typename... A>
struct Call<NUMBER, R(A...)> {
  static inline R (*fn)(A...) = nullptr;
  static PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if constexpr (std::is_integral_v<R>) {
      if (n == static_cast<Py_ssize_t>(sizeof...(A))) return invoke(fn, a, std::index_sequence_for<A...>{});
    }
    Py_RETURN_NOTIMPLEMENTED;
  }
};

#define SGL_AMD_METHOD(number, name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&Call<number, decltype(name)>::call)), METH_FASTCALL, nullptr},
PyMethodDef kCalls[] = {SGL_AMD_NAMES(SGL_AMD_METHOD){nullptr, nullptr, 0, nullptr}};

template <int NUMBER, typename F>
bool found(void* lib, const char* name) {
  using C = Call<NUMBER, F>;
  C::fn = reinterpret_cast<decltype(C::fn)>(dlsym(lib, name));
  return C::fn != nullptr;
}

// bind(path) -> {name: call} of the entry points that the library (loaded already) has
PyObject* bind(PyObject*, PyObject* path) {
  const char* p = PyUnicode_AsUTF8(path);
  if (p == nullptr) return nullptr;
  void* lib = dlopen(p, RTLD_NOW | RTLD_LOCAL);
  if (lib == nullptr) return PyErr_Format(PyExc_OSError, "%s", dlerror());
  PyObject* d = PyDict_New();
  if (d == nullptr) return nullptr;
#define SGL_AMD_BIND(number, name)                                     \
  if (found<number, decltype(name)>(lib, #name)) {                     \
    PyObject* f = PyCFunction_New(&kCalls[number], nullptr);           \
    if (f == nullptr || PyDict_SetItemString(d, #name, f) != 0) {      \
      Py_XDECREF(f);                                                   \
      Py_DECREF(d);                                                    \
      return nullptr;                                                  \
    }                                                                  \
    Py_DECREF(f);                                                      \
  }
  SGL_AMD_NAMES(SGL_AMD_BIND)
  return d;
}

PyMethodDef kMethods[] = {{"bind", bind, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m != nullptr) PyModule_AddStringConstant(m, "header_digest", SGL_AMD_HEADER_DIGEST);
  return m;
}
