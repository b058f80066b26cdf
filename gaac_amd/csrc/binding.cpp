// Python calls of the library's entry points (include/gaac_hip.h): gaac_amd._binding.<entry point>(arguments), raising RuntimeError with the
// library's message where an entry point returns non-zero.  Tensors are handed over as they are; a host tensor raises.  A function in the place of
// an address (the stream) is called for it once the arguments before it have been looked at: without a GPU, a host tensor is what the error names.
// What it is for: a launch has up to 47 arguments, half of them tensors.  Through ctypes, with is_cuda and data_ptr() called from Python for each
// tensor, attention() costs the host 14 us, more than the kernel takes over a short context, and a step of append and attention 24; with the
// arguments converted here 8 to 11 and 12 to 16.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>
#include <exception>
#include <tuple>
#include <type_traits>
#include <utility>
#include "../../include/gaac_hip.h"

namespace {

const char* (*g_last_error)() = nullptr;

// One argument; false with a Python error set.  Numbers convert as ctypes converts them: anything with __index__, cut to the type's bits.
bool convert(PyObject* o, void*& v) {
  if (o == Py_None) { v = nullptr; return true; }
  if (THPVariable_Check(o)) {
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda()) {
      PyErr_SetString(PyExc_RuntimeError, "gaac_amd kernels need device tensors (got a CPU tensor): there is no CPU path");
      return false;
    }
    v = t.data_ptr();
    return true;
  }
  if (PyCallable_Check(o)) {
    PyObject* r = PyObject_CallNoArgs(o);
    const bool ok = r != nullptr && PyLong_Check(r) && convert(r, v);
    if (r != nullptr && !PyLong_Check(r)) PyErr_SetString(PyExc_TypeError, "expected a function that returns an address");
    Py_XDECREF(r);
    return ok;
  }
  if (!PyLong_Check(o)) { PyErr_Format(PyExc_TypeError, "expected a tensor, an address or None, got %s", Py_TYPE(o)->tp_name); return false; }
  v = reinterpret_cast<void*>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
  return !PyErr_Occurred();
}
bool convert(PyObject* o, long& v) {
  if (PyFloat_Check(o)) { PyErr_SetString(PyExc_TypeError, "expected an integer, got float"); return false; }
  v = static_cast<long>(PyLong_AsUnsignedLongMask(o));
  return v != -1 || !PyErr_Occurred();
}
bool convert(PyObject* o, int& v) {
  long l;
  if (!convert(o, l)) return false;
  v = static_cast<int>(l);
  return true;
}
bool convert(PyObject* o, float& v) {
  const double d = PyFloat_AsDouble(o);
  v = static_cast<float>(d);
  return d != -1.0 || !PyErr_Occurred();
}

template <typename A> using Held = std::conditional_t<std::is_pointer_v<A>, void*, A>;      // what an argument is converted to
template <typename A> A passed(Held<A> v) { if constexpr (std::is_pointer_v<A>) return static_cast<A>(v); else return v; }

template <typename... A, size_t... I>
PyObject* invoke(const char* name, int (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
  std::tuple<Held<A>...> held;
  try {
    if (!(convert(args[I], std::get<I>(held)) && ...)) return nullptr;
  } catch (const std::exception& e) {      // a tensor without memory
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(passed<A>(std::get<I>(held))...);
  Py_END_ALLOW_THREADS
  if (rc != 0) {
    PyErr_Format(PyExc_RuntimeError, "%s failed (%d): %s", name, rc, g_last_error());
    return nullptr;
  }
  Py_RETURN_NONE;
}
template <typename... A>
PyObject* invoke(const char* name, int (*fn)(A...), PyObject* const* args, Py_ssize_t n) {
  if (fn == nullptr) { PyErr_SetString(PyExc_RuntimeError, "gaac_amd._binding.bind has not been called"); return nullptr; }
  if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, static_cast<Py_ssize_t>(sizeof...(A)), n);
    return nullptr;
  }
  return invoke(name, fn, args, std::index_sequence_for<A...>{});
}

#define GAAC_ENTRY_POINTS(X)                                                                                                              \
  X(gaac_wait_words) X(gaac_page_finish) X(gaac_cache_check)                                                                              \
  X(gaac_exponent_hist) X(gaac_bases_from_hist) X(gaac_encode_tiles) X(gaac_compact) X(gaac_tile_scan) X(gaac_page_pack)                  \
  X(gaac_row_offsets) X(gaac_decode_tiles) X(gaac_cache_prefill) X(gaac_attn_split) X(gaac_attn_combine) X(gaac_cache_append)             \
  X(gaac_paged_store) X(gaac_paged_free) X(gaac_paged_release) X(gaac_paged_decode) X(gaac_paged_attn) X(gaac_bf16_attn)                  \
  X(gaac_attn_fused) X(gaac_attn_fused_static) X(gaac_static_init) X(gaac_static_reset) X(gaac_static_flags) X(gaac_attn_launch)
#define X(name)                                            \
  decltype(&::name) p_##name = nullptr;                    \
  PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) { return invoke(#name, p_##name, args, n); }
GAAC_ENTRY_POINTS(X)
#undef X

// bind(path): the entry points of the library at path (the product or one of its measurement builds); AttributeError names a missing one
PyObject* bind(PyObject*, PyObject* path) {
  const char* file = PyUnicode_AsUTF8(path);
  if (file == nullptr) return nullptr;
  void* lib = dlopen(file, RTLD_NOW | RTLD_LOCAL);
  if (lib == nullptr) { PyErr_SetString(PyExc_RuntimeError, dlerror()); return nullptr; }
  const auto find = [&](const char* name) {
    void* p = dlsym(lib, name);
    if (p == nullptr && !PyErr_Occurred()) PyErr_Format(PyExc_AttributeError, "%s: undefined symbol: %s", file, name);
    return p;
  };
#define X(name) p_##name = reinterpret_cast<decltype(p_##name)>(find(#name));
  GAAC_ENTRY_POINTS(X)
#undef X
  g_last_error = reinterpret_cast<const char* (*)()>(find("gaac_last_error"));
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

#define X(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {GAAC_ENTRY_POINTS(X){"bind", bind, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
#undef X
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() {
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", GAAC_TORCH_VERSION) != 0) { Py_DECREF(m); return nullptr; }      // whose headers these are
  return m;
}
