// Python extension: calls of a compiled TC on PyTorch tensors, checked and launched natively.
//
// A kernel of a few microseconds is over before an interpreter has looked at its tensors: building
// DLPack descriptors in ctypes took 4 to 6 us per tensor (run() of four tensors 30 us, a call that
// also infers and allocates three results 270 us).  A Plan holds what an executor was compiled on
// (types and sizes of inputs and outputs); its methods read the tensors through ATen, compare them
// with that on every call and launch.  Whatever does not match is left to the general path, which
// reports it: the methods answer False (None) and have launched nothing.
//
//   Plan(executor_handle, error_class)
//   plan.run(inputs, outputs) -> bool            the checks of TcExecutor::run, then the launch
//   plan.unchecked_run(inputs, outputs) -> bool  no checks beyond "these are tensors"
//   plan.call(inputs) -> tensor | tuple | None   run() on results allocated next to inputs[0]
//
// The stream is PyTorch's current one.  Counterpart of tc/aten/aten_compiler.h:69-92 for Python.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <vector>

#include "tc_hip.h"

namespace {

constexpr size_t kMaxTensors = 64;

struct TensorMeta {
  at::ScalarType type = at::ScalarType::Undefined;
  bool byteWide = false; // (uint, 8): one byte per element, a uint8 or a bool tensor
  std::vector<int64_t> sizes;
};

struct Plan {
  PyObject_HEAD
  const tc_executor_t* executor; // owned by the Executor that owns this plan
  std::vector<TensorMeta>* inputs;
  std::vector<TensorMeta>* outputs;
  PyObject* error;
};

at::ScalarType scalarType(const tc_dl_datatype& t) {
  if (t.lanes != 1) return at::ScalarType::Undefined;
  if (t.code == 2) {
    return t.bits == 16 ? at::kHalf : t.bits == 32 ? at::kFloat : t.bits == 64 ? at::kDouble : at::ScalarType::Undefined;
  }
  if (t.code == 0) {
    return t.bits == 8 ? at::kChar : t.bits == 16 ? at::kShort : t.bits == 32 ? at::kInt : t.bits == 64 ? at::kLong : at::ScalarType::Undefined;
  }
  if (t.code == 1) {
    return t.bits == 8 ? at::kByte
        : t.bits == 16 ? at::ScalarType::UInt16
        : t.bits == 32 ? at::ScalarType::UInt32
        : t.bits == 64 ? at::ScalarType::UInt64
                       : at::ScalarType::Undefined;
  }
  return at::ScalarType::Undefined;
}

bool readMetas(const tc_executor_t* executor, int outputs, std::vector<TensorMeta>& metas) {
  const int n = tc_executor_num_tensors(executor, outputs);
  for (int i = 0; i < n; ++i) {
    tc_tensor_info info;
    if (tc_executor_tensor_info(executor, outputs, i, &info) != 0) return false;
    TensorMeta m;
    m.type = scalarType(info.dtype);
    m.byteWide = info.dtype.code == 1 && info.dtype.bits == 8;
    m.sizes.assign(info.shape, info.shape + info.ndim);
    if (m.type == at::ScalarType::Undefined) return false;
    metas.push_back(std::move(m));
  }
  return metas.size() <= kMaxTensors;
}

// Dense row-major tensor of this type and these sizes in the memory of the current device, which is
// asked for (`device` < 0) once a tensor lies on one: a machine without a GPU has none to name.
bool matches(const at::Tensor& t, const TensorMeta& m, c10::DeviceIndex& device) {
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided) return false;
  if (device < 0) device = c10::hip::current_device();
  if (t.get_device() != device) return false;
  if (t.scalar_type() != m.type && !(m.byteWide && t.scalar_type() == at::kBool)) return false;
  return t.sizes() == at::IntArrayRef(m.sizes) && t.is_contiguous() && t.data_ptr() != nullptr;
}

// The items of a list or tuple; false when it is neither.
bool items(PyObject* sequence, PyObject**& first, Py_ssize_t& count) {
  if (PyList_CheckExact(sequence)) {
    first = reinterpret_cast<PyListObject*>(sequence)->ob_item;
    count = PyList_GET_SIZE(sequence);
    return true;
  }
  if (PyTuple_Check(sequence)) {
    first = reinterpret_cast<PyTupleObject*>(sequence)->ob_item;
    count = PyTuple_GET_SIZE(sequence);
    return true;
  }
  return false;
}

using Pointers = std::array<void*, kMaxTensors>;

// Row-major strides in every dimension, those of one element included: is_contiguous() takes any
// stride there, compilation does not, and a defined comprehension compiles on strides it has not seen.
bool hasCanonicalStrides(const at::Tensor& t) {
  const auto sizes = t.sizes(), strides = t.strides();
  int64_t expect = 1;
  for (size_t d = sizes.size(); d-- > 0;) {
    if (strides[d] != expect) return false;
    expect *= sizes[d];
  }
  return true;
}

// data pointers of the tensors when all of them match
bool collect(PyObject* sequence, const std::vector<TensorMeta>& metas, c10::DeviceIndex& device, Pointers& pointers, bool canonical = false) {
  PyObject** first;
  Py_ssize_t count;
  if (!items(sequence, first, count) || static_cast<size_t>(count) != metas.size()) return false;
  for (Py_ssize_t i = 0; i < count; ++i) {
    if (!THPVariable_Check(first[i])) return false;
    const at::Tensor& t = THPVariable_Unpack(first[i]);
    if (!matches(t, metas[i], device) || (canonical && !hasCanonicalStrides(t))) return false;
    pointers[i] = t.data_ptr();
  }
  return true;
}

bool launch(const Plan* plan, const Pointers& in, size_t numIn, const Pointers& out, size_t numOut) {
  void* stream = static_cast<void*>(c10::hip::getCurrentHIPStream().stream());
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = tc_executor_unchecked_run(
      plan->executor, const_cast<const void* const*>(in.data()), static_cast<int>(numIn), const_cast<void* const*>(out.data()),
      static_cast<int>(numOut), stream);
  Py_END_ALLOW_THREADS
  if (status != 0) {
    PyErr_SetString(plan->error, tc_last_error());
    return false;
  }
  return true;
}

PyObject* planRun(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Plan* plan = reinterpret_cast<Plan*>(self);
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "run(inputs, outputs)");
    return nullptr;
  }
  c10::DeviceIndex device = -1;
  Pointers in, out;
  if (!collect(args[0], *plan->inputs, device, in) || !collect(args[1], *plan->outputs, device, out)) Py_RETURN_FALSE;
  if (!launch(plan, in, plan->inputs->size(), out, plan->outputs->size())) return nullptr;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyObject* planUncheckedRun(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Plan* plan = reinterpret_cast<Plan*>(self);
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "unchecked_run(inputs, outputs)");
    return nullptr;
  }
  Pointers pointers[2];
  for (int side = 0; side < 2; ++side) {
    PyObject** first;
    Py_ssize_t count;
    const size_t expected = side == 0 ? plan->inputs->size() : plan->outputs->size();
    if (!items(args[side], first, count) || static_cast<size_t>(count) != expected) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < count; ++i) {
      if (!THPVariable_Check(first[i])) Py_RETURN_FALSE;
      const at::Tensor& t = THPVariable_Unpack(first[i]);
      if (!t.is_cuda()) Py_RETURN_FALSE;
      pointers[side][i] = t.data_ptr();
    }
  }
  if (!launch(plan, pointers[0], plan->inputs->size(), pointers[1], plan->outputs->size())) return nullptr;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyObject* planCall(PyObject* self, PyObject* inputs) {
  HANDLE_TH_ERRORS
  Plan* plan = reinterpret_cast<Plan*>(self);
  if (plan->inputs->empty()) Py_RETURN_NONE;
  c10::DeviceIndex device = -1;
  Pointers in, out;
  if (!collect(inputs, *plan->inputs, device, in, true)) Py_RETURN_NONE;
  std::vector<at::Tensor> results;
  results.reserve(plan->outputs->size());
  for (size_t i = 0; i < plan->outputs->size(); ++i) {
    const TensorMeta& m = (*plan->outputs)[i];
    results.push_back(at::empty(m.sizes, at::TensorOptions().dtype(m.type).device(at::Device(at::kCUDA, device))));
    out[i] = results.back().data_ptr();
    if (out[i] == nullptr) Py_RETURN_NONE;
  }
  if (!launch(plan, in, plan->inputs->size(), out, results.size())) return nullptr;
  if (results.size() == 1) return THPVariable_Wrap(std::move(results[0]));
  PyObject* tuple = PyTuple_New(static_cast<Py_ssize_t>(results.size()));
  if (!tuple) return nullptr;
  for (size_t i = 0; i < results.size(); ++i) {
    PyObject* item = THPVariable_Wrap(std::move(results[i]));
    if (!item) {
      Py_DECREF(tuple);
      return nullptr;
    }
    PyTuple_SET_ITEM(tuple, static_cast<Py_ssize_t>(i), item);
  }
  return tuple;
  END_HANDLE_TH_ERRORS
}

PyObject* planNew(PyTypeObject* type, PyObject* args, PyObject*) {
  unsigned long long handle = 0;
  PyObject* error = nullptr;
  if (!PyArg_ParseTuple(args, "KO", &handle, &error)) return nullptr;
  if (handle == 0) {
    PyErr_SetString(PyExc_ValueError, "null executor");
    return nullptr;
  }
  Plan* self = reinterpret_cast<Plan*>(type->tp_alloc(type, 0));
  if (!self) return nullptr;
  self->executor = reinterpret_cast<const tc_executor_t*>(handle);
  self->inputs = new std::vector<TensorMeta>();
  self->outputs = new std::vector<TensorMeta>();
  Py_INCREF(error);
  self->error = error;
  if (!readMetas(self->executor, 0, *self->inputs) || !readMetas(self->executor, 1, *self->outputs)) {
    Py_DECREF(self);
    PyErr_SetString(PyExc_ValueError, "this executor's tensors have no ATen counterpart");
    return nullptr;
  }
  return reinterpret_cast<PyObject*>(self);
}

void planDealloc(PyObject* object) {
  Plan* self = reinterpret_cast<Plan*>(object);
  delete self->inputs;
  delete self->outputs;
  Py_XDECREF(self->error);
  Py_TYPE(object)->tp_free(object);
}

PyMethodDef planMethods[] = {
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(planRun)), METH_FASTCALL, nullptr},
    {"unchecked_run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(planUncheckedRun)), METH_FASTCALL, nullptr},
    {"call", planCall, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject planType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_call", nullptr, -1, nullptr, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__torch_call(void) {
  planType.tp_name = "_torch_call.Plan";
  planType.tp_basicsize = sizeof(Plan);
  planType.tp_flags = Py_TPFLAGS_DEFAULT;
  planType.tp_new = planNew;
  planType.tp_dealloc = planDealloc;
  planType.tp_methods = planMethods;
  if (PyType_Ready(&planType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&planType);
  if (PyModule_AddObject(m, "Plan", reinterpret_cast<PyObject*>(&planType)) < 0) {
    Py_DECREF(&planType);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
