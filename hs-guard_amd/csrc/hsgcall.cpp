// The C ABI of include/hsg.h as Python functions (CPython extension hs_guard._hsgcall, host code only): every entry point
// that returns a status takes its C arguments positionally (pointers as int addresses or None) and returns the status.
// The argument list of each function comes from its declaration, so the two cannot drift apart. A call of 20 arguments
// costs 0.3 us here against 3 us through ctypes, whose converters run per argument.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/hsg.h"

namespace {

// One C argument from a Python object; on failure the Python error is set (checked once after all arguments).
template <typename T>
T from_py(PyObject* o) {
  if constexpr (std::is_pointer_v<T>) {
    return o == Py_None ? nullptr : reinterpret_cast<T>(PyLong_AsVoidPtr(o));
  } else if constexpr (std::is_floating_point_v<T>) {
    return static_cast<T>(PyFloat_AsDouble(o));
  } else if constexpr (std::is_unsigned_v<T>) {
    return static_cast<T>(PyLong_AsSize_t(o));
  } else {
    const long long v = PyLong_AsLongLong(o);
    if (v != static_cast<T>(v)) PyErr_SetString(PyExc_OverflowError, "integer argument outside its C type");
    return static_cast<T>(v);
  }
}

template <auto Fn, typename... A, size_t... I>
PyObject* invoke(int (*)(A...), PyObject* const* args, std::index_sequence<I...>) {
  std::tuple<A...> c{from_py<A>(args[I])...};
  if (PyErr_Occurred()) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = std::apply(Fn, c);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

template <typename... A>
constexpr size_t arity(int (*)(A...)) {
  return sizeof...(A);
}

template <auto Fn>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  constexpr size_t n = arity(Fn);
  if (nargs != static_cast<Py_ssize_t>(n)) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", static_cast<Py_ssize_t>(n), nargs);
    return nullptr;
  }
  return invoke<Fn>(Fn, args, std::make_index_sequence<n>{});
}

#define HSG_ENTRY(name) \
  { #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&entry<&name>)), METH_FASTCALL, nullptr }

PyMethodDef methods[] = {HSG_ENTRY(hsg_gdn_slot_step),
                         HSG_ENTRY(hsg_gdn_chunk_prefill),
                         HSG_ENTRY(hsg_ring_attention),
                         HSG_ENTRY(hsg_window_attention),
                         HSG_ENTRY(hsg_ring_prefill),
                         HSG_ENTRY(hsg_ring_decode),
                         HSG_ENTRY(hsg_embed_rmsnorm),
                         HSG_ENTRY(hsg_add_rmsnorm),
                         HSG_ENTRY(hsg_gated_rmsnorm),
                         HSG_ENTRY(hsg_conv_silu_update),
                         HSG_ENTRY(hsg_norm_rope),
                         HSG_ENTRY(hsg_add_square),
                         HSG_ENTRY(hsg_rms_finish),
                         HSG_ENTRY(hsg_silu_mul_pair),
                         HSG_ENTRY(hsg_gated_finish),
                         HSG_ENTRY(hsg_square_rows),
                         HSG_ENTRY(hsg_norm_rope_grouped),
                         HSG_ENTRY(hsg_silu_mul),
                         HSG_ENTRY(hsg_risk_head),
                         HSG_ENTRY(hsg_risk_head_f32),
                         HSG_ENTRY(hsg_gdn_slot_step_gated),
                         HSG_ENTRY(hsg_gdn_conv_slot_step_gated),
                         HSG_ENTRY(hsg_gdn_chunk_prefill_gated),
                         HSG_ENTRY(hsg_ring_decode_rope),
                         HSG_ENTRY(hsg_ring_pos_update),
                         HSG_ENTRY(hsg_gemm_bf16),
                         HSG_ENTRY(hsg_gemm_bf16_skinny),
                         HSG_ENTRY(hsg_gemm_bf16_skinny_silu),
                         HSG_ENTRY(hsg_gemm_bf16_skinny_addnorm),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hsgcall", "Entry points of libhsg.so", -1, methods, nullptr, nullptr, nullptr,
                      nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hsgcall(void) { return PyModule_Create(&module); }
