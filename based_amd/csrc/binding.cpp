// The C ABI as Python callables.  ctypes converts arguments one Python object at a time, 2 to 3 us for the forty of an attention call, which is as
// much as a launch; here they are read by the types that include/based_hip.h declares.  What is neither None nor a number in range
// (ctypes arrays, byref) goes to the ctypes entry that a callable was bound with.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "based_hip.h"

namespace {

bool read(PyObject* o, int64_t& x) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  x = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}
bool read(PyObject* o, int& x) {
  int64_t wide = 0;
  if (!read(o, wide) || wide != (int)wide) return false;
  x = (int)wide;
  return true;
}
bool read(PyObject* o, float& x) {
  if (!PyFloat_Check(o)) return false;
  x = (float)PyFloat_AS_DOUBLE(o);
  return true;
}
template <typename P> bool read(PyObject* o, P*& x) {
  int64_t at = 0;
  if (o != Py_None && (!read(o, at) || at < 0)) return false;
  x = reinterpret_cast<P*>(at);
  return true;
}

template <auto F> struct Entry;
template <typename R, typename... A, R (*F)(A...)> struct Entry<F> {
  template <size_t... I> static bool read_all(PyObject* const* args, std::tuple<std::decay_t<A>...>& to, std::index_sequence<I...>) {
    return (read(args[I], std::get<I>(to)) && ...);
  }
  static PyObject* call(PyObject* general, PyObject* const* args, Py_ssize_t n) {
    std::tuple<std::decay_t<A>...> to;
    if (n != (Py_ssize_t)sizeof...(A) || !read_all(args, to, std::index_sequence_for<A...>{})) return PyObject_Vectorcall(general, args, n, nullptr);
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = std::apply(F, to);
    Py_END_ALLOW_THREADS
    return PyLong_FromLongLong((long long)r);
  }
};

struct Listed {
  PyMethodDef def;
  void (*entry)();
};
#define BASED_ENTRY(name)                                                                                                  \
  {{#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<&name>::call)), METH_FASTCALL, nullptr}, \
   reinterpret_cast<void (*)()>(&name)}
Listed kEntries[] = {
    BASED_ENTRY(based_linear_attn_step),
    BASED_ENTRY(based_linear_attn_step_deferred),
    BASED_ENTRY(based_linear_attn_prefill),
    BASED_ENTRY(based_linear_attn_prefill_split),
    BASED_ENTRY(based_linear_attn_prefill_f32),
    BASED_ENTRY(based_swa_prefill),
    BASED_ENTRY(based_swa_prefill_wide),
    BASED_ENTRY(based_swa_step),
    BASED_ENTRY(based_swa_step_wide),
    BASED_ENTRY(based_gated_conv_prefill),
    BASED_ENTRY(based_gated_conv_step),
    BASED_ENTRY(based_short_conv_prefill),
    BASED_ENTRY(based_short_conv_step),
    BASED_ENTRY(based_add_rms_norm),
    BASED_ENTRY(based_swiglu),
    BASED_ENTRY(based_prompt_linear),
    BASED_ENTRY(based_greedy_step),
    BASED_ENTRY(based_decode_linear),
    BASED_ENTRY(based_decode_linear_stream),
    BASED_ENTRY(based_decode_linear_mixes),
    BASED_ENTRY(based_add_norm),
    BASED_ENTRY(based_add_norm_addends),
    BASED_ENTRY(based_stream_conv),
    BASED_ENTRY(based_window_attn_prefill),
    BASED_ENTRY(based_window_attn_attend),
    BASED_ENTRY(based_window_attn_step),
    BASED_ENTRY(based_gated_delta_scan),
    BASED_ENTRY(based_gated_delta_scan_work_of),
    BASED_ENTRY(based_gated_delta_scan_work_as),
    BASED_ENTRY(based_gated_delta_scan_chunks),
    BASED_ENTRY(based_gated_rms_norm),
    BASED_ENTRY(based_gated_delta_step),
    BASED_ENTRY(based_rglru_prefill_work),
    BASED_ENTRY(based_rglru_prefill),
    BASED_ENTRY(based_rglru_step),
    BASED_ENTRY(based_token_mix),
    BASED_ENTRY(based_channel_decay),
    BASED_ENTRY(based_gelu_mul),
    BASED_ENTRY(based_token_side_step),
    BASED_ENTRY(based_softcap),
    BASED_ENTRY(based_decay_scan_work_of),
    BASED_ENTRY(based_decay_scan),
    BASED_ENTRY(based_decay_scan_channels_work),
    BASED_ENTRY(based_decay_scan_channels),
    BASED_ENTRY(based_decay_step),
    BASED_ENTRY(based_group_norm_gate),
    BASED_ENTRY(based_latent_write),
    BASED_ENTRY(based_latent_step),
    BASED_ENTRY(based_expert_tiles),
    BASED_ENTRY(based_expert_tile_rows),
    BASED_ENTRY(based_expert_grouped),
    BASED_ENTRY(based_expert_grouped_f32),
    BASED_ENTRY(based_expert_rows),
};

#ifndef BASED_HIP_INTERFACE
#define BASED_HIP_INTERFACE 0
#endif

// bind(name, address, entry): the callable for an entry point that is listed, the ctypes entry itself for others and for those of another library
// than the one that this is linked to.
PyObject* bind(PyObject*, PyObject* args) {
  const char* name;
  unsigned long long address;
  PyObject* general;
  if (!PyArg_ParseTuple(args, "sKO", &name, &address, &general)) return nullptr;
  for (Listed& e : kEntries)
    if (!std::strcmp(e.def.ml_name, name) && reinterpret_cast<uintptr_t>(e.entry) == address) return PyCFunction_New(&e.def, general);
  Py_INCREF(general);
  return general;
}

// interface(): the number of the header that this was built of
PyObject* interface(PyObject*, PyObject*) { return PyLong_FromLongLong(BASED_HIP_INTERFACE); }

PyMethodDef kModule[] = {{"bind", bind, METH_VARARGS, "bind(name, address, ctypes entry) -> callable"},
                         {"interface", interface, METH_NOARGS, "interface() -> int"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef kDef = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, kModule, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&kDef); }
