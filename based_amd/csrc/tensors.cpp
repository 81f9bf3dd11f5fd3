// What a call into the library asks of its tensors, in one native call each.  Shape, strides, type and device of seven tensors, as a key, take
// Python 1.9 us, and 0.13 here; memory for a result 1.4 us, and 1.0.  Built against one torch, whose version it tells.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

namespace {

PyObject *g_form = nullptr, *g_empty = nullptr;  // the same in Python, for everything that is no ordinary tensor

// A tensor or parameter of torch's own class whose sizes and strides are numbers, and whose memory is its own: no subclass, nothing mapped,
// traced or made functional, not sparse, not nested.
const at::Tensor* ordinary(PyObject* o) {
  if ((PyObject*)Py_TYPE(o) != THPVariableClass && (PyObject*)Py_TYPE(o) != ParameterClass) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  const c10::TensorImpl* impl = t.unsafeGetTensorImpl();
  using c10::DispatchKey;
  static const c10::DispatchKeySet others({DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper, DispatchKey::BatchedNestedTensor,
                                           DispatchKey::Functionalize, DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::NestedTensor});
  if (!t.defined() || impl->has_symbolic_sizes_strides() || impl->key_set().has_any(others) || t.layout() != at::kStrided) return nullptr;
  return &t;
}

// form(*tensors): bytes that are the same for tensors (or None) of the same shapes, strides, types and devices, and for no others.
PyObject* form(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  constexpr int kMost = 384;
  int64_t words[kMost];
  int at = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (args[i] == Py_None) {
      if (at == kMost) return PyObject_Vectorcall(g_form, args, n, nullptr);
      words[at++] = -1;
      continue;
    }
    const at::Tensor* t = ordinary(args[i]);
    if (t == nullptr || at + 1 + 2 * t->dim() > kMost || t->dim() > 255) return PyObject_Vectorcall(g_form, args, n, nullptr);
    const c10::Device device = t->device();
    words[at++] = t->dim() | (int64_t)t->scalar_type() << 8 | (int64_t)(uint8_t)device.type() << 16 | (int64_t)(uint8_t)device.index() << 24;
    for (const int64_t x : t->sizes()) words[at++] = x;
    for (const int64_t x : t->strides()) words[at++] = x;
  }
  return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(words), at * (Py_ssize_t)sizeof(int64_t));
  END_HANDLE_TH_ERRORS
}

// empty(like, dtype, *sizes): a tensor beside `like`.
PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  constexpr Py_ssize_t kMost = 8;
  int64_t sizes[kMost];
  const at::Tensor* like = n >= 2 && n - 2 <= kMost && THPDtype_Check(args[1]) ? ordinary(args[0]) : nullptr;
  bool whole = like != nullptr;
  for (Py_ssize_t i = 2; whole && i < n; ++i) {
    int overflow = 1;
    if (PyLong_CheckExact(args[i])) sizes[i - 2] = PyLong_AsLongLongAndOverflow(args[i], &overflow);
    whole = overflow == 0 && sizes[i - 2] >= 0;
  }
  if (!whole) return PyObject_Vectorcall(g_empty, args, n, nullptr);
  const auto options = at::TensorOptions().device(like->device()).dtype(reinterpret_cast<THPDtype*>(args[1])->scalar_type);
  at::Tensor t;
  {
    pybind11::gil_scoped_release other_threads;
    t = at::empty(at::IntArrayRef(sizes, n - 2), options);
  }
  return THPVariable_Wrap(std::move(t));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kForm = {"form", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&form)), METH_FASTCALL, nullptr};
PyMethodDef kEmpty = {"empty", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&empty)), METH_FASTCALL, nullptr};

// bind(form, empty): both, with what takes the calls that they leave.
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *by_form, *by_empty;
  if (!PyArg_ParseTuple(args, "OO", &by_form, &by_empty)) return nullptr;
  Py_INCREF(by_form);
  Py_INCREF(by_empty);
  Py_XDECREF(g_form);
  Py_XDECREF(g_empty);
  g_form = by_form, g_empty = by_empty;
  PyObject *f = PyCFunction_New(&kForm, nullptr), *e = PyCFunction_New(&kEmpty, nullptr);
  PyObject* both = f != nullptr && e != nullptr ? PyTuple_Pack(2, f, e) : nullptr;
  Py_XDECREF(f);
  Py_XDECREF(e);
  return both;
}

PyObject* torch_version(PyObject*, PyObject*) { return PyUnicode_FromString(TORCH_VERSION); }

PyMethodDef kModule[] = {{"bind", bind, METH_VARARGS, "bind(form, empty) -> the native two"},
                         {"torch_version", torch_version, METH_NOARGS, "torch_version() -> str: the torch that this was built against"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef kDef = {PyModuleDef_HEAD_INIT, "_tensors", nullptr, -1, kModule, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tensors() { return PyModule_Create(&kDef); }
