// deca_amd._launch: the call of a loaded kernel with torch tensors, as one C function.
//
// A kernel of this package is a few microseconds at its smallest (softmax of 256 x 1024: 2.1 us),
// which is less than a Python function takes to check three tensors, ask for the current stream
// and convert six arguments for a foreign-function call.  Here the same steps read torch's own
// structures.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "deca_hip.h"

namespace {

// launch(plan, *tensors): 0 or the hipError_t of the launch on the calling thread's current
// stream; -1, with nothing launched, if an argument is no plain contiguous device tensor or their
// number is not the kernel's (the caller then says which).
PyObject* launch(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n < 1) {
    PyErr_SetString(PyExc_TypeError, "launch(plan, *tensors)");
    return nullptr;
  }
  const auto* plan = static_cast<const deca_plan*>(PyLong_AsVoidPtr(args[0]));
  if (!plan) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "no plan");
    return nullptr;
  }
  if (plan->nargs > 4 || n - 1 != static_cast<Py_ssize_t>(plan->nargs)) return PyLong_FromLong(-1);
  void* ptr[4] = {nullptr, nullptr, nullptr, nullptr};
  try {
    for (Py_ssize_t i = 1; i < n; ++i) {
      if (!THPVariable_CheckExact(args[i])) return PyLong_FromLong(-1);
      const at::Tensor& t = THPVariable_Unpack(args[i]);
      if (!t.is_cuda() || !t.is_contiguous()) return PyLong_FromLong(-1);
      ptr[i - 1] = t.data_ptr();
    }
    void* stream = c10::hip::getCurrentHIPStream().stream();
    int code;
    // (a launch waits where the queue is full: other threads go on meanwhile)
    Py_BEGIN_ALLOW_THREADS
    code = deca_launch_plan(plan, stream, ptr[0], ptr[1], ptr[2], ptr[3]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(code);
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

PyMethodDef methods[] = {
    {"launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(launch)), METH_FASTCALL,
     "launch(plan, *tensors) -> hipError_t, -1 for arguments the kernel cannot take"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// TORCH: the version whose structures `launch` reads; the caller compares it with the one it runs with.
PyMODINIT_FUNC PyInit__launch() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "TORCH", DECA_TORCH) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
