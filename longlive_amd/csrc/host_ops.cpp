// Native host path of the package: the calls a forward is made of, from torch tensors to launches, without Python
// between them.  The kernels and their argument checks are those of the C ABI (include/ll_nvfp4.h); this module
// allocates outputs and temporaries from torch's caching allocator on the tensors' device, takes torch's current
// stream and hands raw pointers on.  In Python the same work costs 20 to 25 us a call (tensor factories, stream and
// device queries, ctypes conversions), more than the kernels of a small call need on the GPU; here it is 2 to 4 us.
//
// Every function returns None for a call it does not take (another device, type, layout or option than the common
// one); the caller then runs the general Python path, which does the work or raises the error that belongs to it.
// Nothing is kept between calls.
#include <Python.h>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/ll_nvfp4.h"

namespace {

using at::Tensor;

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// The index of the tensor's device when that is the current one, else -1 (nothing here may touch the GPU for a tensor
// that is not on it).
inline int current_device_of(const Tensor& t) {
  return t.is_cuda() && t.get_device() == c10::hip::current_device() ? (int)t.get_device() : -1;
}
// A bf16 tensor on that device.
inline bool is_bf16(const Tensor& t, int dev) {
  return t.scalar_type() == at::kBFloat16 && t.is_cuda() && t.get_device() == dev && t.layout() == at::kStrided;
}
inline bool on_device(const Tensor& t, int dev) { return t.is_cuda() && t.get_device() == dev; }

inline Tensor empty(at::IntArrayRef size, at::ScalarType type, int dev) {
  return Tensor(at::detail::empty_cuda(size, type, c10::Device(c10::kCUDA, (c10::DeviceIndex)dev), std::nullopt));
}

inline void* stream_of(int dev) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }

// The codes of the C ABI as the exceptions the Python layer raises for them.
inline bool failed(int code, const char* what) {
  if (code == LL_OK) return false;
  const char* msg = ll_last_error();
  PyErr_SetString(code == LL_EINVAL ? PyExc_ValueError : PyExc_RuntimeError, msg && msg[0] ? msg : what);
  return true;
}

inline const Tensor* as_tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// Python code that traces or redirects torch calls (subclasses, __torch_function__ modes) sees tensors only through
// torch's own functions: such tensors take the general path.
inline bool plain(PyObject* o) { return THPVariable_CheckExact(o); }

PyObject* tuple3(const Tensor& a, const Tensor& b, const Tensor& c) {
  PyObject* r = PyTuple_New(3);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(a));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(b));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(c));
  return r;
}

// A packed NVFP4 operand that lives for one call, in one allocation: values, scales, tensor amax and the partial maxima
// of the amax pass.
struct TempOperand {
  Tensor mem;
  uint8_t* values;
  uint8_t* scales;
  float* amax;
  float* workspace;
  int64_t mp, kp;
};
inline TempOperand temp_operand(int64_t m, int64_t k, int dev) {
  TempOperand t;
  t.mp = round_up(m, 128);
  t.kp = round_up(k, 64);
  const int64_t n_values = t.mp * t.kp / 2, n_scales = t.mp * t.kp / 16;  // multiples of 4096 and 512 bytes
  t.mem = empty({n_values + n_scales + 16 + (int64_t)LL_AMAX_PARTS * 4}, at::kByte, dev);
  t.values = t.mem.data_ptr<uint8_t>();
  t.scales = t.values + n_values;
  t.amax = reinterpret_cast<float*>(t.scales + n_scales);
  t.workspace = t.amax + 4;
  return t;
}

// quantize(x, rule) -> (values, scales, amax): x bf16 [M, K] with contiguous columns.
PyObject* py_quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !plain(args[0])) Py_RETURN_NONE;
  const Tensor& x = THPVariable_Unpack(args[0]);
  const int dev = current_device_of(x);
  if (!is_bf16(x, dev) || x.dim() != 2 || x.stride(1) != 1 || x.numel() == 0) Py_RETURN_NONE;
  const int64_t M = x.size(0), K = x.size(1), Mp = round_up(M, 128), Kp = round_up(K, 64);
  const int rule = (int)PyLong_AsLong(args[1]);
  const Tensor values = empty({Mp, Kp / 2}, at::kByte, dev), scales = empty({Mp * Kp / 16}, at::kFloat8_e4m3fn, dev),
               amax = empty({1}, at::kFloat, dev), ws = empty({(int64_t)LL_AMAX_PARTS}, at::kFloat, dev);
  if (failed(ll_nvfp4_quantize(x.data_ptr(), M, K, x.stride(0), rule, values.data_ptr<uint8_t>(), static_cast<uint8_t*>(scales.data_ptr()),
                               amax.data_ptr<float>(), 0, ws.data_ptr<float>(), stream_of(dev)),
             "ll_nvfp4_quantize"))
    return nullptr;
  return tuple3(values, scales, amax);
  END_HANDLE_TH_ERRORS
}

// linear(x, rule, denom_a, w_values, w_scales, w_amax, denom_b, out_features, bias or None) -> bf16 [M, out_features]:
// activation quantization and GEMM; the operand in between lives for this call.
PyObject* py_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9 || !plain(args[0])) Py_RETURN_NONE;
  const Tensor& x = THPVariable_Unpack(args[0]);
  const Tensor *wv = as_tensor(args[3]), *ws = as_tensor(args[4]), *wa = as_tensor(args[5]), *bias = as_tensor(args[8]);
  const int dev = current_device_of(x);
  if (!wv || !ws || !wa || (!bias && args[8] != Py_None)) Py_RETURN_NONE;
  if (!is_bf16(x, dev) || x.dim() != 2 || x.stride(1) != 1 || x.numel() == 0) Py_RETURN_NONE;
  if (!on_device(*wv, dev) || !on_device(*ws, dev) || !on_device(*wa, dev) || wv->dim() != 2) Py_RETURN_NONE;
  const int64_t M = x.size(0), K = x.size(1), N = PyLong_AsLongLong(args[7]);
  const int rule = (int)PyLong_AsLong(args[1]);
  const double denom_a = PyFloat_AsDouble(args[2]), denom_b = PyFloat_AsDouble(args[6]);
  if (PyErr_Occurred()) return nullptr;
  if (wv->size(1) * 2 != round_up(K, 64) || wv->size(0) != round_up(N, 128) || !wv->is_contiguous() || !ws->is_contiguous()) Py_RETURN_NONE;
  if (bias && (!is_bf16(*bias, dev) || bias->numel() != N || !bias->is_contiguous())) Py_RETURN_NONE;
  void* stream = stream_of(dev);
  const TempOperand a = temp_operand(M, K, dev);
  const Tensor out = empty({M, N}, at::kBFloat16, dev);
  if (failed(ll_nvfp4_quantize(x.data_ptr(), M, K, x.stride(0), rule, a.values, a.scales, a.amax, 0, a.workspace, stream),
             "ll_nvfp4_quantize"))
    return nullptr;
  if (failed(ll_nvfp4_gemm_tnt(a.values, a.scales, wv->data_ptr<uint8_t>(), static_cast<const uint8_t*>(ws->data_ptr()), nullptr,
                               a.amax, wa->data_ptr<float>(), (float)denom_a, (float)denom_b, M, N, a.mp, wv->size(0), a.kp,
                               out.data_ptr(), N, bias ? bias->data_ptr() : nullptr, stream),
             "ll_nvfp4_gemm_tnt"))
    return nullptr;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// dequantize(values, scales, amax, rule, Mp, Kp, M, K, dtype code) -> [M, K]
PyObject* py_dequantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) Py_RETURN_NONE;
  const Tensor *values = as_tensor(args[0]), *scales = as_tensor(args[1]), *amax = as_tensor(args[2]);
  const int dev = values ? current_device_of(*values) : -1;
  if (!values || !scales || !amax || dev < 0 || !on_device(*scales, dev) || !on_device(*amax, dev)) Py_RETURN_NONE;
  int64_t v[6];
  for (int i = 0; i < 6; ++i) v[i] = PyLong_AsLongLong(args[3 + i]);
  if (PyErr_Occurred()) return nullptr;
  const at::ScalarType type = v[5] == LL_DTYPE_BF16 ? at::kBFloat16 : v[5] == LL_DTYPE_F16 ? at::kHalf : at::kFloat;
  const Tensor out = empty({v[3], v[4]}, type, dev);
  if (failed(ll_nvfp4_dequantize(static_cast<const uint8_t*>(values->data_ptr()), static_cast<const uint8_t*>(scales->data_ptr()),
                                 amax->data_ptr<float>(), (int)v[0], v[1], v[2], v[3], v[4], out.data_ptr(), (int)v[5], v[4],
                                 stream_of(dev)),
             "ll_nvfp4_dequantize"))
    return nullptr;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"quantize", (PyCFunction)(void (*)(void))py_quantize, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))py_linear, METH_FASTCALL, nullptr},
    {"dequantize", (PyCFunction)(void (*)(void))py_dequantize, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_ops(void) { return PyModule_Create(&module); }
