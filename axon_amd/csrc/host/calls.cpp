// The kernel library's entry points as Python callables, with the argument types that api.h declares: a launch is one call with
// its numbers read in place.  (ctypes converts and boxes every argument: 2.4 us for the fifteen of a product against 0.36.)
//
// bind(name, address) -> callable: a tensor's address is a whole number or None (or an object whose `value` is one, as ctypes'
// pointers are), everything else a number.  The function runs without the interpreter's lock.  names(): what can be bound.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <string.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "api.h"

#define AXK_CALLS(X) \
  X(axk_embed) X(axk_rmsnorm) X(axk_rope_table) X(axk_rope_kv_write) X(axk_gemm_qkv_rope_ok) X(axk_gemm_qkv_rope) \
  X(axk_gemm_normed_ok) X(axk_gemm_normed_glu) X(axk_gemm_normed_qkv_rope) X(axk_attention) X(axk_attention_prefill) \
  X(axk_attention_decode) X(axk_attention_fast_ok) X(axk_attention_blocks_ok) X(axk_gemm) X(axk_pack_ok) X(axk_pack_matrix) \
  X(axk_gemm_segments) X(axk_gemm_then_norm_ok) X(axk_gemm_then_norm) X(axk_swiglu) X(axk_argmax) X(axk_topk) \
  X(axk_topk_workspace) X(axk_embed_scaled) X(axk_norm_add) X(axk_round_rows) X(axk_activation) X(axk_clamped_glu) \
  X(axk_grouped_gemm_uses_mfma) X(axk_grouped_gemm_by_tile) X(axk_grouped_gemm) X(axk_route_topk) X(axk_route_scored) \
  X(axk_route_max_tiles) X(axk_grouped_gemm_wide) X(axk_route_sort) X(axk_route_combine) X(axk_tanh_norm) X(axk_tanh_norm_add) \
  X(axk_gather_rows) X(axk_causal_conv) X(axk_gated_scan) X(axk_gated_scan_stretches) X(axk_state_conv) X(axk_state_space_scan) \
  X(axk_gated_group_norm) X(axk_token_shift) X(axk_time_mix_decay) X(axk_wkv_scan) X(axk_delta_prepare) X(axk_delta_scan) \
  X(axk_delta_chunked_ok) X(axk_delta_chunked) X(axk_delta_low_rank) X(axk_silu_rows) X(axk_lightning_scan) \
  X(axk_lightning_chunked_ok) X(axk_lightning_chunked) X(axk_embed_pairs) X(axk_scaled_sum) X(axk_shifted_norm) \
  X(axk_head_norm_gate) X(axk_latent_prepare) X(axk_latent_query_rope) X(axk_latent_attention) X(axk_sum_norm) X(axk_layernorm) \
  X(axk_softcap) X(axk_scale_rows) X(axk_add_scaled) X(axk_heads_prepare) X(axk_masked_attention_uses_mfma) \
  X(axk_masked_attention) X(axk_concat_round) X(axk_fill_i32) X(axk_fill_f32) X(axk_attention_decode_workspace) \
  X(axk_gemm_workspace) X(axk_argmax_workspace) X(axk_latent_attention_workspace) X(axk_masked_attention_workspace) \
  X(axk_delta_chunked_workspace)

namespace {

void* address_of(PyObject* o) {
  if (o == Py_None) return nullptr;
  if (PyLong_Check(o)) return PyLong_AsVoidPtr(o);
  PyObject* value = PyObject_GetAttrString(o, "value");
  if (value == nullptr) return nullptr;
  void* p = value == Py_None ? nullptr : PyLong_AsVoidPtr(value);
  Py_DECREF(value);
  return p;
}

template <class T>
T number_of(PyObject* o) {
  if constexpr (std::is_pointer_v<T>) return (T)address_of(o);
  else if constexpr (std::is_floating_point_v<T>) return (T)PyFloat_AsDouble(o);
  else return (T)PyLong_AsLong(o);
}

template <class R, class... A, size_t... I>
PyObject* call_with(R (*f)(A...), PyObject* const* args, std::index_sequence<I...>) {
  const std::tuple<A...> numbers{number_of<A>(args[I])...};
  if (PyErr_Occurred()) return nullptr;
  R result;
  Py_BEGIN_ALLOW_THREADS
  result = f(std::get<I>(numbers)...);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong((long)result);
}

template <class R, class... A>
PyObject* call_as(R (*f)(A...), PyObject* const* args, Py_ssize_t n) {
  if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%zd arguments for an entry point of %zu", n, sizeof...(A));
  return call_with(f, args, std::index_sequence_for<A...>());
}

template <class F>
PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  void* f = PyCapsule_GetPointer(self, nullptr);
  return f == nullptr ? nullptr : call_as((F)f, args, n);
}

#define AXK_ENTRY(NAME) {#NAME, (PyCFunction)(void (*)(void))call<decltype(&NAME)>, METH_FASTCALL, nullptr},
PyMethodDef entries[] = {AXK_CALLS(AXK_ENTRY){nullptr, nullptr, 0, nullptr}};

PyObject* bind(PyObject*, PyObject* args) {
  const char* name;
  unsigned long long address;
  if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
  for (PyMethodDef* e = entries; e->ml_name != nullptr; ++e) {
    if (strcmp(e->ml_name, name) != 0) continue;
    PyObject* capsule = PyCapsule_New((void*)address, nullptr, nullptr);
    if (capsule == nullptr) return nullptr;
    PyObject* callable = PyCFunction_NewEx(e, capsule, nullptr);
    Py_DECREF(capsule);
    return callable;
  }
  return PyErr_Format(PyExc_KeyError, "no entry point %s", name);
}

PyObject* names(PyObject*, PyObject*) {
  PyObject* list = PyList_New(0);
  for (PyMethodDef* e = entries; list != nullptr && e->ml_name != nullptr; ++e) {
    PyObject* name = PyUnicode_FromString(e->ml_name);
    if (name == nullptr || PyList_Append(list, name) != 0) Py_CLEAR(list);
    Py_XDECREF(name);
  }
  return list;
}

PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr}, {"names", names, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "axon_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_axon_calls(void) { return PyModule_Create(&module); }
