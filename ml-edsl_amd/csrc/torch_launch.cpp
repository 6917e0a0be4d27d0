// CPython binding of the device launch entries (include/edsl_hip_device.h) on
// torch tensors: device.dense_launch's operand checks and the call, natively.
//
// The checks read some 25 tensor attributes. Through Python that took 1.85 us of
// the 4.5 us it cost to enqueue a small layer (the library's part, the HIP
// launch included, was the other 2.7), more than the layer itself runs; here
// they take 0.25 us. Three small layers one after another (64 rows through
// 256, 256 and 64 columns): 15.4 us before, 10.6 now; their kernels run 8.4.
//
// dense_launch(X, W, b, Y, epilogue, alpha, stream, current) takes plain
// torch.Tensor objects and Parameters that pass every check, and returns the
// entry's status; anything else -- subclasses, tensors without storage, arguments that a check refuses -- returns
// None before anything is launched, and the caller's Python path handles it or
// names what is wrong. `stream` is the caller's stream object, or None for the
// handle that current() returns; it is asked for after the checks, so that host
// tensors are refused without the GPU being initialised. The GIL is released
// around the call, as in csrc/pylaunch.c.
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/edsl_hip_device.h"

namespace {

// A GPU tensor of this type with unit inner stride.
bool operand_ok(const at::Tensor& t, at::ScalarType type, int64_t dim) {
  if (!t.is_cuda() || t.scalar_type() != type || t.layout() != at::kStrided || t.dim() != dim) return false;
  return t.size(dim - 1) <= 1 || t.stride(dim - 1) == 1;
}

// A conversion failed: the Python path meets the same argument and raises.
PyObject* not_taken() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

PyObject* dense_launch(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 8) {
    PyErr_SetString(PyExc_TypeError, "dense_launch takes 8 arguments");
    return nullptr;
  }
  for (int i : {0, 1, 3})
    if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
  const bool has_bias = args[2] != Py_None;
  if (has_bias && !THPVariable_CheckExact(args[2])) Py_RETURN_NONE;
  const void *x, *w, *b = nullptr;
  void* y;
  int64_t ldx, ldw, ldy, M, N, K;
  bool f32;
  try {
    const at::Tensor &X = THPVariable_Unpack(args[0]), &W = THPVariable_Unpack(args[1]),
                     &Y = THPVariable_Unpack(args[3]);
    const at::ScalarType type = X.scalar_type();
    f32 = type == at::kFloat;
    if (!f32 && type != at::kInt) Py_RETURN_NONE;
    if (!operand_ok(X, type, 2) || !operand_ok(W, type, 2) || !operand_ok(Y, type, 2)) Py_RETURN_NONE;
    M = X.size(0);
    K = X.size(1);
    N = W.size(1);
    if (W.size(0) != K || Y.size(0) != M || Y.size(1) != N) Py_RETURN_NONE;
    if (has_bias) {
      const at::Tensor& B = THPVariable_Unpack(args[2]);
      if (!operand_ok(B, type, 1) || B.size(0) != N) Py_RETURN_NONE;
      b = B.data_ptr();
    }
    x = X.data_ptr();
    w = W.data_ptr();
    y = Y.data_ptr();
    ldx = X.stride(0);
    ldw = W.stride(0);
    ldy = Y.stride(0);
  } catch (...) {  // e.g. a tensor without storage: the Python path raises what it always raised
    Py_RETURN_NONE;
  }
  const long long epilogue = PyLong_AsLongLong(args[4]);
  if (epilogue == -1 && PyErr_Occurred()) return not_taken();
  double alpha = 0.0;
  if (f32) {
    alpha = PyFloat_AsDouble(args[5]);
    if (alpha == -1.0 && PyErr_Occurred()) return not_taken();
  }
  PyObject* handle = args[6] == Py_None ? PyObject_CallNoArgs(args[7]) : PyObject_GetAttrString(args[6], "cuda_stream");
  if (handle == nullptr) return not_taken();
  void* stream = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  if (stream == nullptr && PyErr_Occurred()) return not_taken();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (f32)
    rc = edsl_hip_dense_f32_launch(static_cast<const float*>(x), ldx, static_cast<const float*>(w), ldw,
                                   static_cast<const float*>(b), static_cast<float*>(y), ldy, M, N, K,
                                   static_cast<int>(epilogue), static_cast<float>(alpha), stream);
  else
    rc = edsl_hip_dense_i32_launch(static_cast<const int32_t*>(x), ldx, static_cast<const int32_t*>(w), ldw,
                                   static_cast<const int32_t*>(b), static_cast<int32_t*>(y), ldy, M, N, K,
                                   static_cast<int>(epilogue), stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

PyMethodDef methods[] = {
    {"dense_launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(dense_launch)), METH_FASTCALL,
     "dense_launch(X, W, b, Y, epilogue, alpha, stream, current) -> status, or None when the arguments are not taken"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_launch", "Device launches on torch tensors.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_build names the torch it was compiled against (build.torch_build_id);
// the package uses it with no other.
PyMODINIT_FUNC PyInit__torch_launch(void) {
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_build", EDSL_TORCH_BUILD_ID) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
