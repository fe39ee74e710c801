// CPython entry to the C ABI: one builtin function per entry point the operators call on every layer, taking the same
// arguments in the same order as the C function (integers, floats, None for a null pointer). ctypes spends 6-7 us
// converting the 30-odd arguments of an attention call; this takes under 1 us. The signatures come from the header
// (template deduction), the addresses from the library _lib.py has loaded (bind), so nothing is linked twice. The GIL is
// released around each call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/vox_attn.h"

namespace {

// Pointers from addresses, None or ctypes pointer objects (their `value`); integers reduced to the C type, as ctypes does.
template <typename T>
T convert(PyObject* o) {
  if constexpr (std::is_pointer<T>::value) {
    if (o == Py_None) return nullptr;
    if (PyLong_Check(o)) return (T)PyLong_AsVoidPtr(o);
    PyObject* v = PyObject_GetAttrString(o, "value");
    if (!v) return nullptr;
    T r = v == Py_None ? nullptr : (T)PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    return r;
  } else if constexpr (std::is_floating_point<T>::value) {
    return (T)PyFloat_AsDouble(o);
  } else {
    return (T)PyLong_AsUnsignedLongLongMask(o);
  }
}

template <typename Fn>
struct Entry;
template <typename R, typename... A>
struct Entry<R (*)(A...)> {
  template <std::size_t... I>
  static PyObject* call(R (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v{convert<A>(args[I])...};  // (braces: in order)
    if (PyErr_Occurred()) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = fn(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return std::is_signed<R>::value ? PyLong_FromLongLong((long long)r) : PyLong_FromUnsignedLongLong((unsigned long long)r);
  }
  static PyObject* checked(const char* name, R (*fn)(A...), PyObject* const* args, Py_ssize_t n) {
    if (!fn) {
      PyErr_Format(PyExc_RuntimeError, "%s is not bound", name);
      return nullptr;
    }
    if (n != (Py_ssize_t)sizeof...(A)) {
      PyErr_Format(PyExc_TypeError, "%s takes %zu arguments, got %zd", name, sizeof...(A), n);
      return nullptr;
    }
    return call(fn, args, std::index_sequence_for<A...>{});
  }
};

#define VOX_ENTRIES(X)              \
  X(vox_store_kvcache)              \
  X(vox_decode_attn)                \
  X(vox_decode_attn_store)          \
  X(vox_decode_workgroups)          \
  X(vox_prefill_attn)               \
  X(vox_prefill_attn_store)         \
  X(vox_prefill_attn_store_paged)   \
  X(vox_prefill_attn_int8)          \
  X(vox_prefill_attn_int8_store)    \
  X(vox_prefill_int8_workspace_bytes)

#define VOX_DEFINE(name)                                                              \
  decltype(&name) g_##name = nullptr;                                                 \
  PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) {               \
    return Entry<decltype(&name)>::checked(#name, g_##name, args, n);                 \
  }
VOX_ENTRIES(VOX_DEFINE)

// bind({name: address}): the addresses of the entry points in the loaded library
PyObject* py_bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 1 || !PyDict_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "bind takes one dict");
    return nullptr;
  }
#define VOX_BIND(name)                                                                \
  {                                                                                   \
    PyObject* a = PyDict_GetItemString(args[0], #name);                               \
    if (!a) {                                                                         \
      PyErr_SetString(PyExc_KeyError, #name);                                         \
      return nullptr;                                                                 \
    }                                                                                 \
    g_##name = (decltype(&name))PyLong_AsVoidPtr(a);                                  \
    if (PyErr_Occurred()) return nullptr;                                             \
  }
  VOX_ENTRIES(VOX_BIND)
  Py_RETURN_NONE;
}

#define VOX_METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr},
PyMethodDef methods[] = {VOX_ENTRIES(VOX_METHOD){"bind", (PyCFunction)(void (*)(void))py_bind, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
  PyObject* m = PyModule_Create(&module);
  // the header's version: the signatures above are those of a library of the same one
  if (m && PyModule_AddIntConstant(m, "ABI_VERSION", VOX_ABI_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
