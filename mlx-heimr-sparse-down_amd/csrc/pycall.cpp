// The Python side's calls of libhsd's entry points, without ctypes: one function per entry,
// its argument conversions generated from the entry's own C signature. A pointer argument
// takes None (null), a device tensor (its data pointer), an int or a ctypes pointer. A call of
// 26 arguments costs about 1 us here against 8 us through ctypes, which for a decode step's
// calls was more than their kernels take. The addresses are bound at run time (bind), from
// the library that the Python side has loaded, so this file links to nothing of it.
#include <torch/csrc/autograd/python_variable.h>

#include <exception>
#include <type_traits>

#include "../../include/hsd.h"

namespace {

#define HSD_ENTRIES(X) \
  X(hsd_permute_nibbles) \
  X(hsd_transpose_u16) \
  X(hsd_neuron_major) \
  X(hsd_sparse_down_decode) \
  X(hsd_sparse_down_residual) \
  X(hsd_sparse_down_decode_noalloc) \
  X(hsd_moe_up_relu2) \
  X(hsd_moe_route_up_relu2) \
  X(hsd_router_topk) \
  X(hsd_dense_down_decode) \
  X(hsd_linear) \
  X(hsd_argmax_keys) \
  X(hsd_attn_decode) \
  X(hsd_embed_q4) \
  X(hsd_pair_norm) \
  X(hsd_decode_advance) \
  X(hsd_spec_accept) \
  X(hsd_mtp_chain) \
  X(hsd_seq_select_row) \
  X(hsd_draft_ids) \
  X(hsd_head_input) \
  X(hsd_verify_input) \
  X(hsd_gather_tokens) \
  X(hsd_prefill_advance) \
  X(hsd_seq_rollback) \
  X(hsd_seq_add) \
  X(hsd_rows_prep) \
  X(hsd_gemm_q4) \
  X(hsd_gemm_bf16) \
  X(hsd_moe_tiles) \
  X(hsd_moe_up_gemm) \
  X(hsd_moe_down_gemm) \
  X(hsd_mamba_scan) \
  X(hsd_attn_prompt) \
  X(hsd_kv_append) \
  X(hsd_prompt_tokens) \
  X(hsd_prompt_advance) \
  X(hsd_prefill_tiles) \
  X(hsd_prefill_union) \
  X(hsd_prefill_gemm) \
  X(hsd_mamba_verify) \
  X(hsd_mamba_ssm) \
  X(hsd_mamba_ssm_gated) \
  X(hsd_mamba_select_row) \
  X(hsd_greedy_accept) \
  X(hsd_sparse_down_workspace_bytes) \
  X(hsd_linear_argmax_slots) \
  X(hsd_attn_workspace_bytes) \
  X(hsd_moe_down_workspace_bytes) \
  X(hsd_mamba_scan_workspace_bytes) \
  X(hsd_prefill_num_tiles) \
  X(hsd_prefill_tiles_workspace_bytes) \
  X(hsd_prefill_gemm_workspace_bytes) \
  X(hsd_mamba_workspace_bytes)

enum Entry : int {
#define X(n) k_##n,
  HSD_ENTRIES(X)
#undef X
  kEntries
};

const char* const kNames[] = {
#define X(n) #n,
    HSD_ENTRIES(X)
#undef X
};

void* g_addr[kEntries];
const char* (*g_last_error)() = nullptr;
PyObject* g_error = nullptr;   // the exception class of failed calls

// One argument; false with a Python exception set when it does not convert.
template <typename T>
bool convert(PyObject* o, T& out) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      out = nullptr;
      return true;
    }
    if (THPVariable_Check(o)) {
      const at::Tensor& t = THPVariable_Unpack(o);
      if (!t.is_cuda()) {
        PyErr_SetString(g_error, "libhsd takes device tensors only (got a CPU tensor)");
        return false;
      }
      // a buffer that the entry point writes: a copy-on-write tensor gets memory of its own first
      if constexpr (std::is_const_v<std::remove_pointer_t<T>>)
        out = static_cast<T>(t.const_data_ptr());
      else
        out = static_cast<T>(t.mutable_data_ptr());
      if (!out && t.numel()) {   // a fake tensor: its null would read as "absent"
        PyErr_SetString(g_error, "libhsd takes device tensors only (got a tensor without memory)");
        return false;
      }
      return true;
    }
    if (PyLong_Check(o)) {
      out = reinterpret_cast<T>(PyLong_AsVoidPtr(o));
      return !PyErr_Occurred();
    }
    PyObject* v = PyObject_GetAttrString(o, "value");   // ctypes.c_void_p
    if (v && (v == Py_None || PyLong_Check(v))) {
      out = v == Py_None ? nullptr : reinterpret_cast<T>(PyLong_AsVoidPtr(v));
      Py_DECREF(v);
      return !PyErr_Occurred();
    }
    Py_XDECREF(v);
    PyErr_Clear();
    PyErr_Format(PyExc_TypeError, "a pointer argument takes None, a device tensor, an int or a ctypes pointer, not %s",
                 Py_TYPE(o)->tp_name);
    return false;
  } else if constexpr (std::is_floating_point_v<T>) {
    out = static_cast<T>(PyFloat_AsDouble(o));
    return !PyErr_Occurred();
  } else {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) return false;
    out = static_cast<T>(v);
    if (static_cast<long long>(out) != v) {
      PyErr_SetString(PyExc_OverflowError, "argument out of the C type's range");
      return false;
    }
    return true;
  }
}

// The interpreter's lock given back for a call, and taken again also when it throws.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// An int is a status (0, or an error that is raised); a size is returned.
template <typename R, typename... A, size_t... I>
PyObject* invoke(R (*fn)(A...), const char* name, PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
  if (n != static_cast<Py_ssize_t>(sizeof...(A)))
    return PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, static_cast<Py_ssize_t>(sizeof...(A)), n);
  try {
    std::tuple<A...> a;
    if (!(convert(args[I], std::get<I>(a)) && ...)) return nullptr;
    if constexpr (!std::is_same_v<R, int>) return PyLong_FromLongLong(static_cast<long long>(fn(std::get<I>(a)...)));
    int rc;
    {
      NoGil released;
      rc = static_cast<int>(fn(std::get<I>(a)...));
    }
    if (rc != 0) return PyErr_Format(g_error, "%s -> %d: %s", name, rc, g_last_error());
  } catch (const std::exception& e) {   // a tensor without storage; an entry point out of host memory
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  return PyLong_FromLong(0);
}

template <typename R, typename... A>
PyObject* dispatch(R (*)(A...), int e, PyObject* const* args, Py_ssize_t n) {
  if (!g_addr[e]) return PyErr_Format(PyExc_RuntimeError, "%s is not bound", kNames[e]);
  return invoke(reinterpret_cast<R (*)(A...)>(g_addr[e]), kNames[e], args, n, std::index_sequence_for<A...>{});
}

#define X(n)                                                                        \
  PyObject* call_##n(PyObject*, PyObject* const* args, Py_ssize_t nargs) {          \
    return dispatch(static_cast<decltype(&n)>(nullptr), k_##n, args, nargs);        \
  }
HSD_ENTRIES(X)
#undef X

// bind(exception class, address of hsd_last_error, {entry name: address})
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3 || !PyDict_Check(args[2])) return PyErr_Format(PyExc_TypeError, "bind(error, last_error, addresses)");
  void* le = PyLong_AsVoidPtr(args[1]);
  if (PyErr_Occurred()) return nullptr;
  for (int e = 0; e < kEntries; ++e) {
    PyObject* v = PyDict_GetItemString(args[2], kNames[e]);
    if (!v) return PyErr_Format(PyExc_KeyError, "%s", kNames[e]);
    g_addr[e] = PyLong_AsVoidPtr(v);
    if (PyErr_Occurred()) return nullptr;
  }
  Py_INCREF(args[0]);
  Py_XDECREF(g_error);
  g_error = args[0];
  g_last_error = reinterpret_cast<const char* (*)()>(le);
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL, nullptr},
#define X(n) {#n, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call_##n)), METH_FASTCALL, nullptr},
    HSD_ENTRIES(X)
#undef X
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_hsdcall", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hsdcall() { return PyModule_Create(&kModule); }
