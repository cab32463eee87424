// The address of a torch tensor, for pybind_fast.cpp: the part of the Python front end's call path that needs torch.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/autograd/python_variable.h>

#include <exception>

// 1 and the address, 0 if the object is no tensor, -1 with an exception set
extern "C" __attribute__((visibility("default"))) int pulpnn_tensor_address(PyObject *o, void **out)
try {
  if (!THPVariable_Check(o)) return 0;
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.is_cuda()) {
    PyErr_SetString(PyExc_ValueError, "PULP-NN HIP kernels take device tensors");
    return -1;
  }
  if (!t.is_contiguous()) {
    PyErr_SetString(PyExc_ValueError, "tensor must be contiguous");
    return -1;
  }
  *out = t.data_ptr();
  return 1;
} catch (const std::exception &e) {  // a tensor without storage (a fake or a functional one) has no address
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
  return -1;
}
