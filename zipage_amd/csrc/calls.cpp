// The entry points of the C ABI as Python functions.  A call is the conversion of ten to thirty numbers and addresses, and a launch of
// 2.7 us: 1.2 us less than through ctypes, and a small step makes ten to twenty calls while the GPU waits (a decode step of 8
// requests, two layers of width 1024, 187 -> 171 us; latent attention of 20, 80 -> 72; attention of a prompt of 140 tokens 25 ->
// 22).  Types come from the headers; addresses of the functions from whoever loaded the library.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/zipage_hip.h"
#include "../../include/zipage_models.h"

namespace {

template <class T> bool from(PyObject* o, T& v) {
  if constexpr (std::is_floating_point<T>::value) {
    const double x = PyFloat_AsDouble(o);
    v = (T)x;
    return x != -1.0 || !PyErr_Occurred();
  } else if constexpr (std::is_integral<T>::value) {
    const long long x = PyLong_AsLongLong(o);
    v = (T)x;
    return x != -1 || !PyErr_Occurred();
  } else if (o == Py_None) {
    v = nullptr;
    return true;
  } else if (PyLong_Check(o)) {
    v = (T)PyLong_AsVoidPtr(o);
    return v || !PyErr_Occurred();
  } else {                                       // a ctypes structure or array, or one by reference, which the caller holds
    PyObject* const by = PyObject_CheckBuffer(o) ? nullptr : PyObject_GetAttrString(o, "_obj");
    if (!by) PyErr_Clear();
    Py_buffer b;
    const bool there = PyObject_GetBuffer(by ? by : o, &b, PyBUF_SIMPLE) == 0;
    Py_XDECREF(by);
    if (!there) return false;
    v = (T)b.buf;
    PyBuffer_Release(&b);
    return true;
  }
}

template <class F> struct Entry;
template <class R, class... A> struct Entry<R(A...)> {
  typedef R (*Function)(A...);
  template <size_t... I> static bool convert(PyObject* const* args, std::tuple<A...>& to, std::index_sequence<I...>) {
    return (from(args[I], std::get<I>(to)) && ...);
  }
  // Other threads run while the call does, as under ctypes.
  static PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%zd arguments instead of %zu", n, sizeof...(A));
    std::tuple<A...> values;
    if (!convert(args, values, std::index_sequence_for<A...>())) return nullptr;
    const Function f = (Function)PyCapsule_GetPointer(self, nullptr);
    if (!f) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = std::apply(f, values);
    Py_END_ALLOW_THREADS
    return PyLong_FromLongLong((long long)r);
  }
};

#define ZP_ENTRY(name) {#name, (PyCFunction)(void (*)(void))Entry<decltype(name)>::call, METH_FASTCALL, nullptr}
PyMethodDef entries[] = {
    ZP_ENTRY(zp_store_query), ZP_ENTRY(zp_attention_score), ZP_ENTRY(zp_attention_score_workspace),
    ZP_ENTRY(zp_attention_score_workspace_for), ZP_ENTRY(zp_attention_score_workspace_few), ZP_ENTRY(zp_global_score),
    ZP_ENTRY(zp_pool_scores), ZP_ENTRY(zp_key_norm), ZP_ENTRY(zp_redundancy_lightning), ZP_ENTRY(zp_redundancy_raw),
    ZP_ENTRY(zp_redundancy_raw_workspace), ZP_ENTRY(zp_score_epilogue), ZP_ENTRY(zp_topk_mask), ZP_ENTRY(zp_select_topk),
    ZP_ENTRY(zp_compress_kv), ZP_ENTRY(zp_compress_score), ZP_ENTRY(zp_compress_layers_workspace),
    ZP_ENTRY(zp_compress_layers_workspace_few), ZP_ENTRY(zp_compress_layers), ZP_ENTRY(zp_static_scratch_init),
    ZP_ENTRY(zp_compress_layers_static), ZP_ENTRY(zp_store_kvcache), ZP_ENTRY(zp_paged_decode_attention),
    ZP_ENTRY(zp_paged_decode_workspace), ZP_ENTRY(zp_paged_decode_parts),
    ZP_ENTRY(zp_add_rms_norm), ZP_ENTRY(zp_add_rms_norm_parts), ZP_ENTRY(zp_silu_and_mul), ZP_ENTRY(zp_qk_norm_rope_store), ZP_ENTRY(zp_embed_norm),
    ZP_ENTRY(zp_residual_norm), ZP_ENTRY(zp_normed_powers), ZP_ENTRY(zp_xielu), ZP_ENTRY(zp_relu_square), ZP_ENTRY(zp_softcap),
    ZP_ENTRY(zp_gather_rows), ZP_ENTRY(zp_few_rows_linear), ZP_ENTRY(zp_row_tiles_linear), ZP_ENTRY(zp_split_rows_linear),
    ZP_ENTRY(zp_split_rows_workspace), ZP_ENTRY(zp_run_attention), ZP_ENTRY(zp_causal_attention),
    ZP_ENTRY(zp_latent_norm_store), ZP_ENTRY(zp_rotate_heads), ZP_ENTRY(zp_headwise_linear), ZP_ENTRY(zp_latent_rows_workspace),
    ZP_ENTRY(zp_latent_rows_attention), ZP_ENTRY(zp_rotary_store), ZP_ENTRY(zp_grouped_rows_workspace),
    ZP_ENTRY(zp_grouped_rows_attention), ZP_ENTRY(zp_mlstm_scan), ZP_ENTRY(zp_mlstm_runs_workspace), ZP_ENTRY(zp_mlstm_runs),
    ZP_ENTRY(zp_delta_scan), ZP_ENTRY(zp_delta_runs_workspace), ZP_ENTRY(zp_delta_runs), ZP_ENTRY(zp_linear_scan),
    ZP_ENTRY(zp_linear_runs_workspace), ZP_ENTRY(zp_linear_runs), ZP_ENTRY(zp_small_linear), ZP_ENTRY(zp_moe_select),
    ZP_ENTRY(zp_moe_tile_rows), ZP_ENTRY(zp_moe_max_tiles), ZP_ENTRY(zp_moe_plan_workspace), ZP_ENTRY(zp_moe_plan),
    ZP_ENTRY(zp_moe_gate_up), ZP_ENTRY(zp_moe_down),
};

// entry(name, address): the function at `address`, which is what the headers declare under `name`.
PyObject* entry(PyObject*, PyObject* args) {
  const char* name;
  unsigned long long address;
  if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
  for (PyMethodDef& e : entries) {
    if (std::strcmp(e.ml_name, name) != 0) continue;
    PyObject* const at = PyCapsule_New((void*)address, nullptr, nullptr);
    if (!at) return nullptr;
    PyObject* const f = PyCFunction_New(&e, at);
    Py_DECREF(at);
    return f;
  }
  return PyErr_Format(PyExc_KeyError, "%s", name);
}

PyObject *is_cuda, *data_ptr;
// Address of a device tensor, 0 of None.
PyObject* pointer(PyObject*, PyObject* t) {
  if (t == Py_None) return PyLong_FromLong(0);
  PyObject* const there = PyObject_GetAttr(t, is_cuda);
  if (!there) return nullptr;
  const int yes = PyObject_IsTrue(there);
  Py_DECREF(there);
  if (yes < 0) return nullptr;
  if (!yes) {
    PyErr_SetString(PyExc_RuntimeError, "the compression kernels need device tensors (no CPU fallback)");
    return nullptr;
  }
  return PyObject_CallMethodNoArgs(t, data_ptr);
}

PyMethodDef methods[] = {{"entry", entry, METH_VARARGS, nullptr}, {"pointer", pointer, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "zipage_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_zipage_calls() {
  is_cuda = PyUnicode_InternFromString("is_cuda");
  data_ptr = PyUnicode_InternFromString("data_ptr");
  return is_cuda && data_ptr ? PyModule_Create(&module) : nullptr;
}
