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

PyObject *held_types, *pointer_types, *cast, *void_pointer;      // of ctypes
// Where a ctypes structure, union or array lies, or what a ctypes pointer or reference points to; the caller holds it.  Nothing else
// that has a buffer: a NumPy number would pass its own address.  `record`: bytes of the structure that is wanted, 0: any.
bool address(PyObject* o, void*& v, size_t record) {
  const int held = PyObject_IsInstance(o, held_types), other = held ? 0 : PyObject_IsInstance(o, pointer_types);
  if (held < 0 || other < 0) return false;
  if (!held && !other) return PyErr_Format(PyExc_TypeError, "%s in a pointer's place", Py_TYPE(o)->tp_name), false;
  PyObject* to = o;
  if (other) {
    PyObject* const p = PyObject_CallFunctionObjArgs(cast, o, void_pointer, nullptr);
    if (!p) return false;
    PyObject* const value = PyObject_GetAttrString(p, "value");
    Py_DECREF(p);
    if (!value) return false;
    v = value == Py_None ? nullptr : PyLong_AsVoidPtr(value);
    Py_DECREF(value);
    if (!v && PyErr_Occurred()) return false;
    if (!record) return true;
    to = PyObject_GetAttrString(o, "_obj");
    if (!to) return PyErr_Format(PyExc_TypeError, "%s in a structure's place", Py_TYPE(o)->tp_name), false;
  }
  Py_buffer b;
  const bool there = PyObject_GetBuffer(to, &b, PyBUF_SIMPLE) == 0;
  if (other) Py_DECREF(to);
  if (!there) return false;
  const size_t bytes = (size_t)b.len;
  if (held) v = b.buf;
  PyBuffer_Release(&b);
  if (record && (bytes == 0 || bytes % record)) return PyErr_Format(PyExc_TypeError, "%zu bytes instead of a structure's %zu", bytes, record), false;
  return true;
}

template <class T> constexpr size_t record_bytes() {
  if constexpr (std::is_class<T>::value) return sizeof(T);
  else return 0;
}
template <class T> bool from(PyObject* o, T& v) {
  if constexpr (std::is_floating_point<T>::value) {
    const double x = PyFloat_AsDouble(o);
    v = (T)x;
    return x != -1.0 || !PyErr_Occurred();
  } else if constexpr (std::is_integral<T>::value) {
    const long long x = PyLong_AsLongLong(o);
    v = (T)x;
    return x != -1 || !PyErr_Occurred();
  } else {
    constexpr size_t record = record_bytes<std::remove_cv_t<std::remove_pointer_t<T>>>();
    if (o == Py_None) {
      v = nullptr;
      return true;
    }
    if (!record && PyLong_Check(o)) {
      v = (T)PyLong_AsVoidPtr(o);
      return v || !PyErr_Occurred();
    }
    void* at = nullptr;
    const bool there = address(o, at, record);
    v = (T)at;
    return there;
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
    ZP_ENTRY(zp_delta_scan), ZP_ENTRY(zp_delta_runs_workspace), ZP_ENTRY(zp_delta_runs), ZP_ENTRY(zp_delta_runs_projected), ZP_ENTRY(zp_linear_scan),
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

#ifndef ZP_PYTHON
#define ZP_TEXT_OF(x) #x
#define ZP_TEXT(x) ZP_TEXT_OF(x)
#define ZP_PYTHON ZP_TEXT(PY_MAJOR_VERSION) "." ZP_TEXT(PY_MINOR_VERSION) "."
#endif
constexpr char kPython[] = ZP_PYTHON;

PyMethodDef methods[] = {{"entry", entry, METH_VARARGS, nullptr}, {"pointer", pointer, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "zipage_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_zipage_calls() {
  // objects are laid out as in the Python that this was compiled against
  if (std::strncmp(Py_GetVersion(), kPython, sizeof(kPython) - 1) != 0)
    return PyErr_Format(PyExc_ImportError, "libzipage_calls.so is for Python %sx, this is %.20s: build it again", kPython, Py_GetVersion());
  is_cuda = PyUnicode_InternFromString("is_cuda");
  data_ptr = PyUnicode_InternFromString("data_ptr");
  PyObject* const ctypes = PyImport_ImportModule("ctypes");
  PyObject* const inner = ctypes ? PyImport_ImportModule("_ctypes") : nullptr;
  if (!inner) return nullptr;
  cast = PyObject_GetAttrString(ctypes, "cast");
  void_pointer = PyObject_GetAttrString(ctypes, "c_void_p");
  PyObject* const some = void_pointer ? PyObject_CallNoArgs(void_pointer) : nullptr;
  PyObject* const by = some ? PyObject_CallMethod(ctypes, "byref", "O", some) : nullptr;
  if (!cast || !by) return nullptr;
  held_types = Py_BuildValue("(NNN)", PyObject_GetAttrString(ctypes, "Structure"), PyObject_GetAttrString(ctypes, "Union"),
                             PyObject_GetAttrString(ctypes, "Array"));
  pointer_types = Py_BuildValue("(NNOO)", PyObject_GetAttrString(inner, "_Pointer"), PyObject_GetAttrString(inner, "CFuncPtr"), void_pointer,
                                (PyObject*)Py_TYPE(by));
  Py_DECREF(by);
  Py_DECREF(some);
  Py_DECREF(inner);
  Py_DECREF(ctypes);
  return held_types && pointer_types && is_cuda && data_ptr ? PyModule_Create(&module) : nullptr;
}
