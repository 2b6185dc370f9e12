// The host's part of a call that is all launch: Python module ringattn_calls, used by api.py.
//
// A forward of a few hundred tokens, or one step of a short ring, is some 5 us of GPU work, and a launch costs the host 4.3 us of
// its own.  The checks of five tensors, their addresses and the stream took Python another 2.2 (6.8 us a call of forward()); here they take
// 0.2 (4.4).  A Call holds one entry point of the C ABI with its plan and the shapes and types it expects.  Called with five tensors and a stream it
// returns the entry point's code, or None, without having done anything, where the arguments are not plainly what it
// expects: the caller then goes the general way, which says what is wrong, or serves what is merely unusual (tensor subclasses).
// Only addresses of this call's tensors are handed on; nothing of a tensor is kept.
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstddef>
#include <new>
#include <vector>

namespace {

constexpr int kTensors = 5;
using Fwd = int (*)(void*, const void*, const void*, const void*, void*, void*, void*);
using Step = int (*)(void*, int, int, const void*, const void*, const void*, void*, void*, void*);

struct Spec {
  at::ScalarType type;
  std::vector<int64_t> shape;
};
struct Call {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  void* entry;
  void* plan;
  int rank, step;  // rank < 0: an entry point without them
  std::vector<Spec>* specs;
};

PyObject* call(PyObject* self_, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  Call* self = reinterpret_cast<Call*>(self_);
  if (PyVectorcall_NARGS(nargsf) != kTensors + 1 || kwnames) {
    PyErr_SetString(PyExc_TypeError, "five tensors and a stream (or None)");
    return nullptr;
  }
  void* p[kTensors];
  hipStream_t stream;
  try {
    for (int i = 0; i < kTensors; ++i) {
      if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
      const at::Tensor& t = THPVariable_Unpack(args[i]);
      const Spec& s = (*self->specs)[i];
      if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || t.scalar_type() != s.type || t.sizes() != s.shape || !t.is_contiguous())
        Py_RETURN_NONE;
      p[i] = t.data_ptr();
    }
    if (args[kTensors] == Py_None) stream = c10::hip::getCurrentHIPStream().stream();
  } catch (...) {  // a tensor without storage, or whose sizes are symbols
    Py_RETURN_NONE;
  }
  if (args[kTensors] != Py_None) {
    PyObject* handle = PyObject_GetAttrString(args[kTensors], "cuda_stream");
    if (!handle) return nullptr;
    stream = static_cast<hipStream_t>(PyLong_AsVoidPtr(handle));
    Py_DECREF(handle);
    if (PyErr_Occurred()) return nullptr;
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (self->rank < 0) rc = reinterpret_cast<Fwd>(self->entry)(self->plan, p[0], p[1], p[2], p[3], p[4], stream);
  else rc = reinterpret_cast<Step>(self->entry)(self->plan, self->rank, self->step, p[0], p[1], p[2], p[3], p[4], stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// Call(address of the entry point, of the plan, rank or -1, step, ((dtype, shape), ... of five tensors))
PyObject* create(PyTypeObject* type, PyObject* args, PyObject* kwargs) {
  unsigned long long entry, plan;
  int rank, step;
  PyObject* specs;
  if (kwargs && PyDict_Size(kwargs) > 0) {
    PyErr_SetString(PyExc_TypeError, "positional arguments only");
    return nullptr;
  }
  if (!PyArg_ParseTuple(args, "KKiiO!", &entry, &plan, &rank, &step, &PyTuple_Type, &specs)) return nullptr;
  if (!entry || PyTuple_GET_SIZE(specs) != kTensors) {
    PyErr_SetString(PyExc_ValueError, "an entry point and five tensors' types and shapes");
    return nullptr;
  }
  Call* self = reinterpret_cast<Call*>(type->tp_alloc(type, 0));
  if (!self) return nullptr;
  self->vectorcall = call;
  self->entry = reinterpret_cast<void*>(static_cast<uintptr_t>(entry));
  self->plan = reinterpret_cast<void*>(static_cast<uintptr_t>(plan));
  self->rank = rank;
  self->step = step;
  try {
    self->specs = new std::vector<Spec>(kTensors);
    for (int i = 0; i < kTensors; ++i) {
      PyObject *dtype, *shape;
      if (!PyArg_ParseTuple(PyTuple_GET_ITEM(specs, i), "OO!", &dtype, &PyTuple_Type, &shape) || !THPDtype_Check(dtype)) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "a torch.dtype and a tuple");
        Py_DECREF(self);
        return nullptr;
      }
      Spec& s = (*self->specs)[i];
      s.type = reinterpret_cast<THPDtype*>(dtype)->scalar_type;
      for (Py_ssize_t j = 0; j < PyTuple_GET_SIZE(shape); ++j) s.shape.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(shape, j)));
      if (PyErr_Occurred()) {
        Py_DECREF(self);
        return nullptr;
      }
    }
  } catch (const std::bad_alloc&) {
    Py_DECREF(self);
    return PyErr_NoMemory();
  }
  return reinterpret_cast<PyObject*>(self);
}

void destroy(PyObject* self) {
  delete reinterpret_cast<Call*>(self)->specs;
  Py_TYPE(self)->tp_free(self);
}

PyTypeObject call_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "ringattn_calls", "checks and launch of a call", -1};

}  // namespace

PyMODINIT_FUNC PyInit_ringattn_calls() {
  call_type.tp_name = "ringattn_calls.Call";
  call_type.tp_basicsize = sizeof(Call);
  call_type.tp_dealloc = destroy;
  call_type.tp_vectorcall_offset = offsetof(Call, vectorcall);
  call_type.tp_call = PyVectorcall_Call;
  call_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  call_type.tp_new = create;
  if (PyType_Ready(&call_type) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&call_type);
  if (PyModule_AddObject(m, "Call", reinterpret_cast<PyObject*>(&call_type)) < 0) {
    Py_DECREF(&call_type);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
