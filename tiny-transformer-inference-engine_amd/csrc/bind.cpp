// Python calls into libpagedkv.so without ctypes: every entry point of
// include/pagedkv.h as a vectorcall function of the module _pkvbind, its
// arguments converted by the C signature (None is a null pointer). A ctypes call
// with the attention's 29 arguments costs about 4 us, as much as the small
// kernels behind it; these cost under 1. The addresses come from the loaded
// library (bind()), so both ways reach the same instance. As with ctypes, the
// interpreter lock is released during the call. Only the stable ABI is used, so
// one build serves every CPython from 3.10 on; where the module is not there the
// wrappers call through ctypes (serving/_native.py).
#define Py_LIMITED_API 0x030A0000
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/pagedkv.h"

namespace {

// One argument as the C type A; a Python error is left set when it does not fit.
template <typename A>
A convert(PyObject* o) {
  if constexpr (std::is_pointer_v<A>) {
    if (o == Py_None) return nullptr;
    return static_cast<A>(PyLong_AsVoidPtr(o));
  } else if constexpr (std::is_floating_point_v<A>) {
    return static_cast<A>(PyFloat_AsDouble(o));
  } else if constexpr (std::is_same_v<A, size_t>) {
    return PyLong_AsSize_t(o);
  } else {
    const long long v = PyLong_AsLongLong(o);
    const A a = static_cast<A>(v);
    if (static_cast<long long>(a) != v && !PyErr_Occurred())
      PyErr_Format(PyExc_OverflowError, "argument %lld does not fit a C int", v);
    return a;
  }
}

template <typename R, typename... A, size_t... I>
PyObject* invoke(R (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
  const std::tuple<A...> t{convert<A>(args[I])...};  // in order, left to right
  if (PyErr_Occurred()) return nullptr;
  R r;
  Py_BEGIN_ALLOW_THREADS;
  r = std::apply(fn, t);
  Py_END_ALLOW_THREADS;
  if constexpr (std::is_same_v<R, const char*>) return PyBytes_FromString(r ? r : "");
  else if constexpr (std::is_unsigned_v<R>) return PyLong_FromUnsignedLongLong(r);
  else return PyLong_FromLongLong(r);
}

template <typename R, typename... A>
PyObject* checked(const char* name, R (*fn)(A...), PyObject* const* args, Py_ssize_t n) {
  if (!fn) {
    PyErr_Format(PyExc_RuntimeError, "%s: bind() has not been called", name);
    return nullptr;
  }
  if (n != (Py_ssize_t)sizeof...(A)) {
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name,
                 (Py_ssize_t)sizeof...(A), n);
    return nullptr;
  }
  return invoke(fn, args, std::index_sequence_for<A...>{});
}

#define PKV_ENTRIES(X)                                                                       \
  X(pkv_version) X(pkv_append) X(pkv_append_from_table) X(pkv_gather)                        \
  X(pkv_attention_workspace_bytes) X(pkv_paged_attention) X(pkv_paged_attention_append)      \
  X(pkv_paged_attention_noalloc) X(pkv_rms_norm) X(pkv_rope) X(pkv_silu_mul) X(pkv_linear)   \
  X(pkv_linear_swiglu) X(pkv_linear_rope_qkv) X(pkv_linear_residual)                         \
  X(pkv_linear_swiglu_rmsnorm) X(pkv_linear_rope_qkv_rmsnorm) X(pkv_linear_tiles)            \
  X(pkv_linear_tiles_rope_qkv) X(pkv_argmax_rows) X(pkv_sample_rows)                         \
  X(pkv_argmax_workspace_bytes) X(pkv_stream_read)

#define DEFINE(name)                                                                         \
  decltype(&::name) ptr_##name = nullptr;                                                    \
  PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) {                      \
    return checked(#name, ptr_##name, args, n);                                              \
  }
PKV_ENTRIES(DEFINE)
#undef DEFINE

// bind({name: address}): the library's entry points.
PyObject* py_bind(PyObject*, PyObject* table) {
  if (!PyDict_Check(table)) {
    PyErr_SetString(PyExc_TypeError, "bind takes a dict of addresses");
    return nullptr;
  }
#define BIND(name)                                                                           \
  {                                                                                          \
    PyObject* o = PyDict_GetItemString(table, #name);                                        \
    void* p = o ? PyLong_AsVoidPtr(o) : nullptr;                                             \
    if (!p) {                                                                                \
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);                         \
      return nullptr;                                                                        \
    }                                                                                        \
    std::memcpy(&ptr_##name, &p, sizeof(p));                                                 \
  }
  PKV_ENTRIES(BIND)
#undef BIND
  Py_RETURN_NONE;
}

#define METHOD(name)                                                                         \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)),            \
   METH_FASTCALL, nullptr},
PyMethodDef methods[] = {PKV_ENTRIES(METHOD){"bind", py_bind, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
#undef METHOD

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pkvbind", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pkvbind(void) { return PyModule_Create(&module); }
