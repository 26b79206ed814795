// Native host path of the package: the calls a forward is made of, from torch tensors to launches, without Python
// between them.  The kernels and their argument checks are those of the C ABI (include/ll_nvfp4.h); this module
// allocates outputs and temporaries from torch's caching allocator on the tensors' device, takes torch's current
// stream and hands raw pointers on.  In Python the same work costs 20 to 25 us a call (tensor factories, stream and
// device queries, ctypes conversions), more than the kernels of a small call need on the GPU; here it is 2 to 4 us.
//
// A transformer block is one call too (block_forward, 21 launches): issued one by one from Python it took 600 us of host
// time, more than the GPU needs for a block of up to about 2000 tokens.
//
// Every function returns None for a call it does not take (another device, type, layout or option than the common
// one); the caller then runs the general Python path, which does the work or raises the error that belongs to it.
// Nothing is kept between calls but one amax sink (8 KB) per device and stream, which release_stream_memory gives back.
#include <Python.h>

#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/linear.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <map>
#include <mutex>
#include <utility>

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

// ------------------------------------------------------------------------------------------------ amax sinks
// The sink through which the kernels of one native call hand tensor maxima on belongs to the (device, stream) pair: launches
// on one stream are ordered, and two streams (or the threads that drive them) never meet in one buffer.
struct StreamSink {
  Tensor parts;
  uint32_t epoch = 0;
};
std::mutex g_sink_mutex;
std::map<std::pair<int, void*>, StreamSink>& stream_sinks() {
  static auto* sinks = new std::map<std::pair<int, void*>, StreamSink>;  // outlives every static that may still hold tensors
  return *sinks;
}
constexpr uint32_t kEpochsPerCall = 16;

// Epochs for the producers of one call, in the order in which they run.
struct Epochs {
  uint64_t* parts;
  const uint32_t* offset;
  uint32_t next;
  ll_amax_sink take() { return ll_amax_sink{parts, ++next, offset}; }
};
// A failing query (the legacy stream while another one is captured) counts as recording, and leaves no error behind.
bool recording(void* stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(static_cast<hipStream_t>(stream), &status) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return status != hipStreamCaptureStatusNone;
}

// parts is null while the stream is being captured: a recorded epoch would be the same in every replay, whose maxima the
// slots, raised meanwhile by later epochs, would then hide.
Epochs epochs_of_stream(int dev, void* stream) {
  if (recording(stream)) return Epochs{nullptr, nullptr, 0};
  std::lock_guard<std::mutex> lock(g_sink_mutex);
  auto& sinks = stream_sinks();
  const std::pair<int, void*> key{dev, stream};
  auto found = sinks.find(key);
  if (found == sinks.end() || found->second.epoch > 0xFFFFFF00u) {
    if (found == sinks.end()) found = sinks.emplace(key, StreamSink{empty({(int64_t)LL_AMAX_PARTS}, at::kLong, dev), 0}).first;
    // not through torch's zero_: it may have a mode to report to, or refuse a tensor made in inference mode
    if (hipMemsetAsync(found->second.parts.data_ptr(), 0, LL_AMAX_PARTS * sizeof(uint64_t),
                       static_cast<hipStream_t>(stream)) != hipSuccess) {
      (void)hipGetLastError();
      sinks.erase(found);
      return Epochs{nullptr, nullptr, 0};
    }
    found->second.epoch = 0;
  }
  StreamSink& s = found->second;
  const Epochs e{reinterpret_cast<uint64_t*>(s.parts.data_ptr<int64_t>()), nullptr, s.epoch};
  s.epoch += kEpochsPerCall;
  return e;
}

// The amax of x and its quantization: one launch for a small tensor, two otherwise and while the stream is being captured.
// workspace: LL_AMAX_PARTS floats, or null: allocated where two launches need them (1173 x 2048 in one launch: 8.9, so 8.4 us of host time a call).
// The line: two tiles per workgroup and one workgroup per unit for all tensors together.  With two workgroups per unit the
// launch is ahead only where it is repeated by itself (2 x 408 tiles 10.7 against 12.3 us).  Behind an attention launch, as in
// a KV step, it is not; us, two launches / one, by tiles of K and of V: 192 (768 queries x 16 heads) 28.4 / 27.9, 256 (1024 x 16)
// 33.5 / 32.3, 288 (1152 x 16) 38.5 / 39.8, 384 (1536 x 16) 46.8 / 49.4, 288 (768 x 24, 1536 cached) 55.1 / 57.8.
inline bool one_pass_tiles(int64_t M, int64_t K, int tensors) { return K % 64 == 0 && tensors * ((M + 127) / 128) * (K / 64) <= 512; }
int quantize_operand(const void* x, int64_t M, int64_t K, int64_t ldx, int rule, uint8_t* values, uint8_t* scales, float* amax,
                     float* workspace, int dev, void* stream) {
  if (one_pass_tiles(M, K, 1)) {
    Epochs e = epochs_of_stream(dev, stream);
    if (e.parts) {
      const ll_amax_sink sink = e.take();
      const int code = ll_nvfp4_quantize_one_pass(x, nullptr, M, K, ldx, rule, values, nullptr, scales, nullptr, amax, nullptr, &sink,
                                                  LL_EXCHANGE_LOOKS, stream);
      if (code != LL_ENOSUP) return code;
    }
  }
  Tensor own;  // freed for work behind this launch on the stream
  if (!workspace) {
    own = empty({(int64_t)LL_AMAX_PARTS}, at::kFloat, dev);
    workspace = own.data_ptr<float>();
  }
  return ll_nvfp4_quantize(x, M, K, ldx, rule, values, scales, amax, 0, workspace, stream);
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
               amax = empty({1}, at::kFloat, dev);
  if (failed(quantize_operand(x.data_ptr(), M, K, x.stride(0), rule, values.data_ptr<uint8_t>(),
                              static_cast<uint8_t*>(scales.data_ptr()), amax.data_ptr<float>(), nullptr, dev, stream_of(dev)),
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
  if (wv->size(1) * 2 != round_up(K, 64) || wv->size(0) != round_up(N, 128) || !wv->is_contiguous() || !ws->is_contiguous())
    Py_RETURN_NONE;
  if (bias && (!is_bf16(*bias, dev) || bias->numel() != N || !bias->is_contiguous())) Py_RETURN_NONE;
  void* stream = stream_of(dev);
  const Tensor out = empty({M, N}, at::kBFloat16, dev);
  ll_gemm_epilogue epilogue{};
  epilogue.bias = bias ? bias->data_ptr() : nullptr;
  const int code = ll_nvfp4_quantize_gemm(x.data_ptr(), M, K, x.stride(0), rule, nullptr, (float)denom_a, wv->data_ptr<uint8_t>(),
                                          static_cast<const uint8_t*>(ws->data_ptr()), wa->data_ptr<float>(), (float)denom_b, N,
                                          wv->size(0), out.data_ptr(), N, &epilogue, stream);
  if (code != LL_ENOSUP) {
    if (failed(code, "ll_nvfp4_quantize_gemm")) return nullptr;
    return THPVariable_Wrap(out);
  }
  const TempOperand a = temp_operand(M, K, dev);
  if (failed(quantize_operand(x.data_ptr(), M, K, x.stride(0), rule, a.values, a.scales, a.amax, a.workspace, dev, stream),
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

// ------------------------------------------------------------------------------------------------ block
struct Layer {  // a quantized linear layer
  const uint8_t *values, *scales;
  const float* amax;
  const void* bias;
  float denom;
  int64_t np, kp, n;
};
// From (values, scale_factors, amax, bias or None, denominator, out_features); false: not for this path.
bool parse_layer(PyObject* t, int dev, Layer& l) {
  if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != 6) return false;
  const Tensor *v = as_tensor(PyTuple_GET_ITEM(t, 0)), *s = as_tensor(PyTuple_GET_ITEM(t, 1)), *a = as_tensor(PyTuple_GET_ITEM(t, 2));
  PyObject* b = PyTuple_GET_ITEM(t, 3);
  const Tensor* bias = as_tensor(b);
  if (!v || !s || !a || (!bias && b != Py_None)) return false;
  if (!on_device(*v, dev) || !on_device(*s, dev) || !on_device(*a, dev) || v->dim() != 2 || !v->is_contiguous() ||
      !s->is_contiguous())
    return false;
  l.n = PyLong_AsLongLong(PyTuple_GET_ITEM(t, 5));
  l.np = v->size(0);
  l.kp = v->size(1) * 2;
  if (l.np != round_up(l.n, 128) || l.n % 8) return false;
  if (bias && (!is_bf16(*bias, dev) || bias->numel() != l.n || !bias->is_contiguous())) return false;
  l.values = v->data_ptr<uint8_t>();
  l.scales = static_cast<const uint8_t*>(s->data_ptr());
  l.amax = a->data_ptr<float>();
  l.bias = bias ? bias->data_ptr() : nullptr;
  l.denom = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(t, 4));
  return true;
}
// The attended slots: (table of the K slots, of the V slots, cached keys, block_token_size, e2m1_max, e4m3_max) or None.
struct Window {
  const uint64_t* p[6] = {};  // K values, scales, amax, then V
  int64_t n_cached = 0;
  int bts = 0;
  float e2 = 6.f, e4 = 256.f;
};
bool parse_window(PyObject* o, int dev, Window& w) {
  if (o == Py_None) return true;
  if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 6) return false;
  for (int i = 0; i < 2; ++i) {
    const Tensor* t = as_tensor(PyTuple_GET_ITEM(o, i));
    if (!t || !on_device(*t, dev) || t->scalar_type() != at::kLong || t->dim() != 2 || t->size(0) != 3 || !t->is_contiguous())
      return false;
    for (int j = 0; j < 3; ++j) w.p[3 * i + j] = reinterpret_cast<const uint64_t*>(t->data_ptr<int64_t>()) + j * t->size(1);
  }
  w.n_cached = PyLong_AsLongLong(PyTuple_GET_ITEM(o, 2));
  w.bts = (int)PyLong_AsLong(PyTuple_GET_ITEM(o, 3));
  w.e2 = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(o, 4));
  w.e4 = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(o, 5));
  return !PyErr_Occurred();
}

// A (parts, epoch) tuple as a sink; false: not one.
bool parse_sink(PyObject* t, int dev, ll_amax_sink& s) {
  const Tensor* parts = PyTuple_CheckExact(t) && PyTuple_GET_SIZE(t) == 2 ? as_tensor(PyTuple_GET_ITEM(t, 0)) : nullptr;
  if (!parts || !on_device(*parts, dev)) return false;
  s = ll_amax_sink{reinterpret_cast<uint64_t*>(parts->data_ptr<int64_t>()),
                   (uint32_t)PyLong_AsUnsignedLong(PyTuple_GET_ITEM(t, 1)), nullptr};
  return !PyErr_Occurred();
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

struct BlockCall {
  int dev, rule;
  float denom_a;
  void* stream;
  int64_t L, C;

  // out = epilogue(a @ layer^T)
  int gemm(const TempOperand& a, const Layer& w, int64_t M, void* out, ll_gemm_epilogue e) const {
    e.bias = w.bias;
    return ll_nvfp4_gemm_tnt_fused(a.values, a.scales, w.values, w.scales, nullptr, a.amax, w.amax, denom_a, w.denom, M, w.n,
                                   a.mp, w.np, a.kp, out, w.n, &e, stream);
  }
  // out = epilogue(x @ layer^T), the maximum of x in `sink`: one launch for small activations, else quantization into q and product
  int linear(const void* x, int64_t K, const ll_amax_sink& sink, const Layer& w, int64_t M, void* out, ll_gemm_epilogue e, TempOperand& q) const {
    e.bias = w.bias;
    const int code = ll_nvfp4_quantize_gemm(x, M, K, K, rule, &sink, denom_a, w.values, w.scales, w.amax, w.denom, w.n, w.np, out, w.n, &e,
                                            stream);
    if (code != LL_ENOSUP) return code;
    if (!q.values) q = operand(M, K);
    const int quantized = ll_nvfp4_quantize_from_sink(x, M, K, K, rule, q.values, q.scales, q.amax, &sink, stream);
    return quantized ? quantized : gemm(q, w, M, out, e);
  }
  static void products(const Layer* const* w, int n, void* const* outs, const ll_amax_sink* sinks, ll_gemm_product* p) {
    for (int i = 0; i < n; ++i)
      p[i] = ll_gemm_product{w[i]->values, w[i]->scales, nullptr, w[i]->amax, w[i]->denom, outs[i], w[i]->n, w[i]->bias,
                             sinks ? sinks[i] : ll_amax_sink{nullptr, 0, nullptr}};
  }
  int grouped(const TempOperand& a, const Layer* const* w, int n, int64_t M, void* const* outs, const ll_amax_sink* sinks) const {
    ll_gemm_product p[4];
    products(w, n, outs, sinks, p);
    return ll_nvfp4_gemm_tnt_grouped(a.values, a.scales, a.amax, denom_a, M, w[0]->n, a.mp, w[0]->np, a.kp, n, p, stream);
  }
  TempOperand operand(int64_t m, int64_t k) const { return temp_operand(m, k, dev); }
  int quantize_from(const Tensor& x, int64_t M, int64_t K, const TempOperand& q, const ll_amax_sink& sink) const {
    return ll_nvfp4_quantize_from_sink(x.data_ptr(), M, K, K, rule, q.values, q.scales, q.amax, &sink, stream);
  }
};

// block_forward(x, e, layers, norms, cos, sin, kv, text, options, k_sink, v_sink, graph_sink) ->
//   (x_out or None, roped K [1, L, H, 128], V [1, L, H, 128], text K, text V) or None
//   e: the six modulation vectors per frame [1, F, 6, C];  layers: q, k, v, o, cross q, k, v, o, FFN up, down;  norms: weights of
//   norm_q, norm_k, norm3, norm3's bias, cross norm_q, cross norm_k;  kv: the window (see Window);  text: the context [1, T, C]
//   or (K, V) [1, T, H, 128];  options: (rule, denominator, heads, eps, eps of q/k norm, of norm3, of cross norm_q, of cross
//   norm_k, spin limit, keys_only);  k_sink, v_sink: (parts, epoch) or None;  graph_sink: (parts, last epoch, offset) or None.
// The launches and their order are those of DiTBlock.forward (longlive_amd/dit/model.py), which documents them.
PyObject* py_block_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12 || !plain(args[0]) || !plain(args[1])) Py_RETURN_NONE;
  const Tensor& x = THPVariable_Unpack(args[0]);
  const Tensor& e = THPVariable_Unpack(args[1]);
  const int dev = current_device_of(x);
  if (!is_bf16(x, dev) || !is_bf16(e, dev) || x.dim() != 3 || x.size(0) != 1 || !x.is_contiguous() || e.dim() != 4 || e.size(0) != 1 ||
      e.size(2) != 6 || e.size(3) != x.size(2) || e.stride(3) != 1)
    Py_RETURN_NONE;
  BlockCall c;
  c.dev = dev;
  c.L = x.size(1);
  c.C = x.size(2);
  const int64_t L = c.L, C = c.C, F = e.size(1);
  if (L == 0 || F == 0 || L % F || C % 128 || e.stride(1) % 8 || e.stride(2) % 8 || !aligned16(e.data_ptr()) ||
      !aligned16(x.data_ptr()))
    Py_RETURN_NONE;
  const int64_t frame_rows = L / F;
  if (!PyTuple_CheckExact(args[2]) || PyTuple_GET_SIZE(args[2]) != 10 || !PyTuple_CheckExact(args[3]) ||
      PyTuple_GET_SIZE(args[3]) != 6 || !PyTuple_CheckExact(args[8]) || PyTuple_GET_SIZE(args[8]) != 10)
    Py_RETURN_NONE;
  Layer w[10];
  for (int i = 0; i < 10; ++i)
    if (!parse_layer(PyTuple_GET_ITEM(args[2], i), dev, w[i])) Py_RETURN_NONE;
  enum { Q, K, V, O, CQ, CK, CV, CO, UP, DOWN };
  for (int i = 0; i < 10; ++i)
    if (w[i].kp != round_up(i == DOWN ? w[UP].n : C, 64) || (i != UP && w[i].n != C)) Py_RETURN_NONE;
  const void* norm[6];
  for (int i = 0; i < 6; ++i) {
    const Tensor* t = as_tensor(PyTuple_GET_ITEM(args[3], i));
    if (!t || !is_bf16(*t, dev) || t->numel() != C || !t->is_contiguous() || !aligned16(t->data_ptr())) Py_RETURN_NONE;
    norm[i] = t->data_ptr();
  }
  const Tensor *cos = as_tensor(args[4]), *sin = as_tensor(args[5]);
  if (!cos || !sin || !on_device(*cos, dev) || !on_device(*sin, dev) || cos->scalar_type() != at::kFloat ||
      sin->scalar_type() != at::kFloat || !cos->is_contiguous() || !sin->is_contiguous() || cos->numel() != L * 64 ||
      sin->numel() != L * 64)
    Py_RETURN_NONE;
  PyObject* const o = args[8];
  c.rule = (int)PyLong_AsLong(PyTuple_GET_ITEM(o, 0));
  c.denom_a = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(o, 1));
  const int H = (int)PyLong_AsLong(PyTuple_GET_ITEM(o, 2));
  float eps[5];
  for (int i = 0; i < 5; ++i) eps[i] = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(o, 3 + i));
  const int64_t spin = PyLong_AsLongLong(PyTuple_GET_ITEM(o, 8));
  const bool keys_only = PyObject_IsTrue(PyTuple_GET_ITEM(o, 9)) == 1;
  if (PyErr_Occurred()) return nullptr;
  if ((int64_t)H * 128 != C) Py_RETURN_NONE;
  Window kv;
  if (!parse_window(args[6], dev, kv)) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
  // the text: its context, or the projected keys and values
  const Tensor* context = as_tensor(args[7]);
  Tensor text_k, text_v;
  int64_t T = 0;
  if (context) {
    if (!is_bf16(*context, dev) || context->dim() != 3 || context->size(0) != 1 || context->size(2) != C || !context->is_contiguous() ||
        context->size(1) == 0)
      Py_RETURN_NONE;
    T = context->size(1);
  } else {
    if (!PyTuple_CheckExact(args[7]) || PyTuple_GET_SIZE(args[7]) != 2) Py_RETURN_NONE;
    const Tensor *tk = as_tensor(PyTuple_GET_ITEM(args[7], 0)), *tv = as_tensor(PyTuple_GET_ITEM(args[7], 1));
    if (!tk || !tv || !is_bf16(*tk, dev) || !is_bf16(*tv, dev) || !tk->is_contiguous() || !tv->is_contiguous() || tk->dim() != 4 ||
        tk->sizes() != tv->sizes() || tk->size(0) != 1 || tk->size(2) != H || tk->size(3) != 128 || tk->size(1) == 0)
      Py_RETURN_NONE;
    text_k = *tk;
    text_v = *tv;
    T = tk->size(1);
  }
  ll_amax_sink kv_sink[2] = {{nullptr, 0, nullptr}, {nullptr, 0, nullptr}};
  for (int i = 0; i < 2; ++i)
    if (args[9 + i] != Py_None && !parse_sink(args[9 + i], dev, kv_sink[i])) {
      if (PyErr_Occurred()) return nullptr;
      Py_RETURN_NONE;
    }
  c.stream = stream_of(dev);
  Epochs ep;
  if (args[11] == Py_None) {
    ep = epochs_of_stream(dev, c.stream);
    if (!ep.parts) Py_RETURN_NONE;
  } else {
    PyObject* t = args[11];
    const Tensor *parts = as_tensor(PyTuple_GET_ITEM(t, 0)), *offset = as_tensor(PyTuple_GET_ITEM(t, 2));
    if (!parts || !offset || !on_device(*parts, dev) || !on_device(*offset, dev)) Py_RETURN_NONE;
    ep = Epochs{reinterpret_cast<uint64_t*>(parts->data_ptr<int64_t>()), reinterpret_cast<const uint32_t*>(offset->data_ptr<int32_t>()),
                (uint32_t)PyLong_AsUnsignedLong(PyTuple_GET_ITEM(t, 1))};
    if (PyErr_Occurred()) return nullptr;
  }
#define LL_TRY(call, what) \
  if (failed(call, what)) return nullptr

  const uint16_t* mod = static_cast<const uint16_t*>(e.data_ptr());
  const int64_t sb = e.stride(0), sf = e.stride(1);
  auto modulation = [&](int i) { return mod + i * e.stride(2); };
  // LayerNorm(h) * (1 + e[scale]) + e[shift] as an NVFP4 operand: one launch, or two where the rows do not fit one
  auto adaln_operand = [&](const void* h, int scale, int shift, const TempOperand& q, const ll_amax_sink& sink) -> int {
    int code = ll_adaln_quantize(h, 1, L, (int)C, modulation(scale), modulation(shift), sb, sf, sb, sf, frame_rows, eps[0], 1, c.rule,
                                 q.values, q.scales, q.amax, &sink, spin, c.stream);
    if (code != LL_ENOSUP) return code;
    const ll_amax_sink again = ep.take();
    const Tensor y = empty({L, C}, at::kBFloat16, dev);
    code = ll_adaln_modulate_amax(h, 1, L, (int)C, modulation(scale), modulation(shift), sb, sf, sb, sf, frame_rows, eps[0], 1,
                                  y.data_ptr(), &again, c.stream);
    return code ? code : c.quantize_from(y, L, C, q, again);
  };
  // The layers behind a normalization of h [L, C] (adaLN with the modulation vectors `scale` and `shift`, or norm3 where scale is
  // negative) in one launch, for small activations.  LL_ENOSUP, as for every wider block: nothing is launched, `exchange` is unused.
  auto norm_gemm = [&](const void* h, int scale, int shift, const ll_amax_sink& exchange, const Layer* const* layers, int n, void* const* outs,
                       const ll_amax_sink* sinks, int activation, const ll_row_norm* row_norms, float row_eps) -> int {
    if (C > LL_NORM_GEMM_MAX_C) return LL_ENOSUP;
    ll_gemm_product p[4];
    BlockCall::products(layers, n, outs, sinks, p);
    const bool adaln = scale >= 0;
    return ll_nvfp4_norm_gemm(h, L, (int)C, adaln ? modulation(scale) : nullptr, adaln ? modulation(shift) : nullptr, sf, sf, frame_rows, 1,
                              adaln ? nullptr : norm[2], adaln ? nullptr : norm[3], adaln ? eps[0] : eps[2], c.rule, &exchange, spin,
                              c.denom_a, layers[0]->n, layers[0]->np, n, p, activation, row_norms, row_eps, cos->data_ptr<float>(),
                              sin->data_ptr<float>(), L, c.stream);
  };
  TempOperand xq{};  // allocated by the first that needs it

  // ---- self-attention
  const Tensor value = empty({1, L, H, 128}, at::kBFloat16, dev), key = empty({1, L, H, 128}, at::kBFloat16, dev);
  Tensor attended;  // [L, C]
  ll_amax_sink attended_sink;
  {
    const Tensor roped_q = empty({L, C}, at::kBFloat16, dev), smooth_k = empty({L, C}, at::kBFloat16, dev);
    const Layer* const layers[3] = {&w[Q], &w[K], &w[V]};
    void* const normed[3] = {roped_q.data_ptr(), key.data_ptr(), value.data_ptr()};
    const ll_row_norm row_norms[3] = {{norm[0], nullptr, 1}, {norm[1], smooth_k.data_ptr(), 1}, {nullptr, nullptr, 0}};
    const ll_amax_sink exchange = ep.take(), normed_sinks[3] = {{nullptr, 0, nullptr}, kv_sink[0], kv_sink[1]};
    int code = norm_gemm(x.data_ptr(), 1, 0, exchange, layers, 3, normed, normed_sinks, LL_ACT_NONE, row_norms, eps[1]);
    if (code == LL_ENOSUP) {
      const Tensor q = empty({L, C}, at::kBFloat16, dev), k = empty({L, C}, at::kBFloat16, dev);
      void* const outs[3] = {q.data_ptr(), k.data_ptr(), value.data_ptr()};
      const ll_amax_sink sinks[3] = {{nullptr, 0, nullptr}, {nullptr, 0, nullptr}, kv_sink[1]};
      xq = c.operand(L, C);
      LL_TRY(adaln_operand(x.data_ptr(), 1, 0, xq, exchange), "adaLN");
      LL_TRY(c.grouped(xq, layers, 3, L, outs, sinks), "q / k / v projections");
      code = ll_qk_norm_rope_pair_amax(q.data_ptr(), k.data_ptr(), L, H, norm[0], norm[1], eps[1], cos->data_ptr<float>(), sin->data_ptr<float>(),
                                       L, roped_q.data_ptr(), key.data_ptr(), smooth_k.data_ptr(), &kv_sink[0], c.stream);
    }
    LL_TRY(code, "q / k / v projections, norm and RoPE");
    if (keys_only) {
      PyObject* r = PyTuple_New(5);
      if (!r) return nullptr;
      for (int i : {0, 3, 4}) {
        Py_INCREF(Py_None);
        PyTuple_SET_ITEM(r, i, Py_None);
      }
      PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(key));
      PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(value));
      return r;
    }
    attended = empty({L, C}, at::kBFloat16, dev);
    attended_sink = ep.take();
    LL_TRY(ll_kv_attention_amax(roped_q.data_ptr(), L, H, kv.p[0], kv.p[1], kv.p[2], kv.p[3], kv.p[4], kv.p[5], kv.n_cached,
                                kv.bts, kv.e2, kv.e4, smooth_k.data_ptr(), value.data_ptr(), L, 0.08838834764831845f,
                                attended.data_ptr(), &attended_sink, c.stream), "self-attention");
  }
  const Tensor x1 = empty({1, L, C}, at::kBFloat16, dev);
  ll_gemm_epilogue plain_epilogue{}, gated{};
  gated.gate_rows = frame_rows;
  gated.gate_stride = sf;
  gated.ldr = C;
  gated.gate = modulation(2);
  gated.residual = x.data_ptr();
  LL_TRY(c.linear(attended.data_ptr(), C, attended_sink, w[O], L, x1.data_ptr(), gated, xq), "output projection");

  // ---- cross-attention
  auto norm3_operand = [&](const ll_amax_sink& sink) -> int {
    int code = ll_layer_norm_quantize(x1.data_ptr(), L, (int)C, norm[2], norm[3], eps[2], c.rule, xq.values, xq.scales, xq.amax, &sink, spin,
                                      c.stream);
    if (code != LL_ENOSUP) return code;
    const ll_amax_sink again = ep.take();
    const Tensor y = empty({L, C}, at::kBFloat16, dev);
    code = ll_layer_norm(x1.data_ptr(), L, (int)C, norm[2], norm[3], eps[2], y.data_ptr(), &again, c.stream);
    return code ? code : c.quantize_from(y, L, C, xq, again);
  };
  {
    const Tensor qn = empty({L, C}, at::kBFloat16, dev);
    const Layer* const layers[1] = {&w[CQ]};
    void* const normed[1] = {qn.data_ptr()};
    const ll_row_norm row_norms[1] = {{norm[4], nullptr, 0}};
    const ll_amax_sink exchange = ep.take();
    int code = norm_gemm(x1.data_ptr(), -1, -1, exchange, layers, 1, normed, nullptr, LL_ACT_NONE, row_norms, eps[3]);
    if (code == LL_ENOSUP) {
      const Tensor q = empty({L, C}, at::kBFloat16, dev);
      if (!xq.values) xq = c.operand(L, C);
      LL_TRY(norm3_operand(exchange), "norm3");
      LL_TRY(c.gemm(xq, w[CQ], L, q.data_ptr(), plain_epilogue), "cross-attention q");
      code = ll_rms_norm(q.data_ptr(), L, (int)C, norm[4], eps[3], qn.data_ptr(), c.stream);
    }
    LL_TRY(code, "cross-attention q");
    if (context) {
      const TempOperand tq = c.operand(T, C);
      code = LL_ENOSUP;
      if (one_pass_tiles(T, C, 1)) {  // a block of 736 rows, text of 512 x 1536: in two launches 237.2 us, so 234.4
        const ll_amax_sink sink = ep.take();
        code = ll_nvfp4_quantize_one_pass(context->data_ptr(), nullptr, T, C, C, c.rule, tq.values, nullptr, tq.scales, nullptr, tq.amax, nullptr,
                                          &sink, spin, c.stream);
      }
      if (code == LL_ENOSUP)
        code = ll_nvfp4_quantize(context->data_ptr(), T, C, C, c.rule, tq.values, tq.scales, tq.amax, 0, tq.workspace, c.stream);
      LL_TRY(code, "text quantization");
      const Tensor k = empty({T, C}, at::kBFloat16, dev);
      text_k = empty({1, T, H, 128}, at::kBFloat16, dev);
      text_v = empty({1, T, H, 128}, at::kBFloat16, dev);
      const Layer* const layers[2] = {&w[CK], &w[CV]};
      void* const outs[2] = {k.data_ptr(), text_v.data_ptr()};
      LL_TRY(c.grouped(tq, layers, 2, T, outs, nullptr), "text projections");
      LL_TRY(ll_rms_norm(k.data_ptr(), T, (int)C, norm[5], eps[4], text_k.data_ptr(), c.stream), "cross-attention norm_k");
    }
    attended_sink = ep.take();
    LL_TRY(ll_kv_attention_amax(qn.data_ptr(), L, H, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 6.f, 256.f,
                                text_k.data_ptr(), text_v.data_ptr(), T, 0.08838834764831845f, attended.data_ptr(), &attended_sink,
                                c.stream),
           "cross-attention");
  }
  const Tensor x2 = empty({1, L, C}, at::kBFloat16, dev);
  ll_gemm_epilogue residual{};
  residual.ldr = C;
  residual.residual = x1.data_ptr();
  LL_TRY(c.linear(attended.data_ptr(), C, attended_sink, w[CO], L, x2.data_ptr(), residual, xq), "cross-attention output projection");

  // ---- feed-forward
  const Tensor hidden = empty({L, w[UP].n}, at::kBFloat16, dev);
  ll_gemm_epilogue gelu{};
  gelu.activation = LL_ACT_GELU_TANH;
  {
    const Layer* const layers[1] = {&w[UP]};
    void* const outs[1] = {hidden.data_ptr()};
    const ll_amax_sink exchange = ep.take();
    gelu.amax_sink = ep.take();  // newer than the exchange, and below newer than what adaLN may take behind it
    int code = norm_gemm(x2.data_ptr(), 4, 3, exchange, layers, 1, outs, &gelu.amax_sink, LL_ACT_GELU_TANH, nullptr, 0.f);
    if (code == LL_ENOSUP) {
      if (!xq.values) xq = c.operand(L, C);
      LL_TRY(adaln_operand(x2.data_ptr(), 4, 3, xq, exchange), "adaLN");
      gelu.amax_sink = ep.take();
      code = c.gemm(xq, w[UP], L, hidden.data_ptr(), gelu);
    }
    LL_TRY(code, "FFN up");
  }
  TempOperand hq{};
  const Tensor& out = attended;  // its memory is free by now
  gated.gate = modulation(5);
  gated.residual = x2.data_ptr();
  LL_TRY(c.linear(hidden.data_ptr(), w[UP].n, gelu.amax_sink, w[DOWN], L, out.data_ptr(), gated, hq), "FFN down");
#undef LL_TRY

  PyObject* r = PyTuple_New(5);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(out.view({1, L, C})));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(key));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(value));
  PyTuple_SET_ITEM(r, 3, THPVariable_Wrap(text_k));
  PyTuple_SET_ITEM(r, 4, THPVariable_Wrap(text_v));
  return r;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ KV-cache step
// A contiguous bf16 [1, tokens, H, 128] tensor of plain torch type on that device.
const Tensor* as_chunk(PyObject* o, int dev) {
  if (!plain(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  const bool ok = is_bf16(t, dev) && t.dim() == 4 && t.size(0) == 1 && t.size(3) == 128 && t.numel() > 0 && t.is_contiguous() &&
                  aligned16(t.data_ptr());
  return ok ? &t : nullptr;
}

// slot_addresses(K slots, V slots, ids) -> the addresses of the values, scale_factors and amax buffers of those slots of either
// list, packed: what a pointer table of the window is found by (24 buffers for four slots, 3 us in Python).
PyObject* py_slot_addresses(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  static PyObject* const names[3] = {PyUnicode_InternFromString("values"), PyUnicode_InternFromString("scale_factors"),
                                     PyUnicode_InternFromString("amax")};
  if (n != 3 || !PyList_CheckExact(args[0]) || !PyList_CheckExact(args[1]) || !PyTuple_CheckExact(args[2])) Py_RETURN_NONE;
  const Py_ssize_t ids = PyTuple_GET_SIZE(args[2]);
  PyObject* key = PyBytes_FromStringAndSize(nullptr, ids * 2 * 3 * (Py_ssize_t)sizeof(void*));
  if (!key) return nullptr;
  void** out = reinterpret_cast<void**>(PyBytes_AS_STRING(key));
  for (int side = 0; side < 2; ++side)
    for (Py_ssize_t i = 0; i < ids; ++i) {
      const Py_ssize_t at = PyLong_AsSsize_t(PyTuple_GET_ITEM(args[2], i));
      if (at < 0 || at >= PyList_GET_SIZE(args[side])) {
        Py_DECREF(key);
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
      }
      for (PyObject* name : names) {
        PyObject* t = PyObject_GetAttr(PyList_GET_ITEM(args[side], at), name);
        const bool tensor = t && THPVariable_Check(t) && THPVariable_Unpack(t).has_storage();
        if (tensor) *out++ = THPVariable_Unpack(t).data_ptr();
        Py_XDECREF(t);
        if (!tensor) {
          Py_DECREF(key);
          if (PyErr_Occurred()) return nullptr;
          Py_RETURN_NONE;
        }
      }
    }
  return key;
  END_HANDLE_TH_ERRORS
}

// kv_attention(q, k, v, smoothed K or None, window, scale) -> [1, S, H, 128]
PyObject* py_kv_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6 || !plain(args[0])) Py_RETURN_NONE;
  const int dev = current_device_of(THPVariable_Unpack(args[0]));
  if (dev < 0) Py_RETURN_NONE;
  const Tensor *q = as_chunk(args[0], dev), *k = as_chunk(args[1], dev), *v = as_chunk(args[2], dev);
  if (!q || !k || !v || k->sizes() != v->sizes() || k->size(2) != q->size(2)) Py_RETURN_NONE;
  const int H = (int)q->size(2);
  Tensor smooth;
  if (args[3] != Py_None) {
    const Tensor* s = as_chunk(args[3], dev);
    if (!s || s->sizes() != k->sizes()) Py_RETURN_NONE;
    smooth = *s;
  }
  Window w;
  if (!parse_window(args[4], dev, w)) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
  const float scale = (float)PyFloat_AsDouble(args[5]);
  if (PyErr_Occurred()) return nullptr;
  void* stream = stream_of(dev);
  if (!smooth.defined()) {
    smooth = empty(k->sizes(), at::kBFloat16, dev);
    if (failed(ll_kv_smooth(k->data_ptr(), k->size(1), H, smooth.data_ptr(), stream), "ll_kv_smooth")) return nullptr;
  }
  const Tensor out = empty(q->sizes(), at::kBFloat16, dev);
  if (failed(ll_kv_attention(q->data_ptr(), q->size(1), H, w.p[0], w.p[1], w.p[2], w.p[3], w.p[4], w.p[5], w.n_cached, w.bts,
                             w.e2, w.e4, smooth.data_ptr(), v->data_ptr(), k->size(1), scale, out.data_ptr(), stream),
             "ll_kv_attention"))
    return nullptr;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// kv_attention_relative(q, k, v, window, cos_k, sin_k, cos_q, sin_q, scale) -> [1, S, H, 128]
PyObject* py_kv_attention_relative(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9 || !plain(args[0])) Py_RETURN_NONE;
  const int dev = current_device_of(THPVariable_Unpack(args[0]));
  if (dev < 0) Py_RETURN_NONE;
  const Tensor *q = as_chunk(args[0], dev), *k = as_chunk(args[1], dev), *v = as_chunk(args[2], dev);
  if (!q || !k || !v || k->sizes() != v->sizes() || k->sizes() != q->sizes()) Py_RETURN_NONE;
  const int H = (int)q->size(2);
  const int64_t S = q->size(1);
  Window w;
  if (!parse_window(args[3], dev, w)) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
  const int64_t keys = w.n_cached + S;
  const float* tables[4];
  for (int i = 0; i < 4; ++i) {
    const Tensor* t = as_tensor(args[4 + i]);
    if (!t || !on_device(*t, dev) || t->scalar_type() != at::kFloat || !t->is_contiguous() || t->numel() != (i < 2 ? keys : S) * 64 ||
        !aligned16(t->data_ptr()))
      Py_RETURN_NONE;
    tables[i] = t->data_ptr<float>();
  }
  const float scale = (float)PyFloat_AsDouble(args[8]);
  if (PyErr_Occurred()) return nullptr;
  void* stream = stream_of(dev);
  const Tensor wk = empty({keys, H, 128}, at::kBFloat16, dev), wv = empty({keys, H, 128}, at::kBFloat16, dev);
  const Tensor rq = empty(q->sizes(), at::kBFloat16, dev), out = empty(q->sizes(), at::kBFloat16, dev);
  if (failed(ll_kv_window_rope(q->data_ptr(), S, H, w.p[0], w.p[1], w.p[2], w.p[3], w.p[4], w.p[5], w.n_cached, w.bts, w.e2,
                               w.e4, k->data_ptr(), v->data_ptr(), S, tables[0], tables[1], tables[2], tables[3],
                               rq.data_ptr(), wk.data_ptr(), wv.data_ptr(), stream), "ll_kv_window_rope"))
    return nullptr;
  if (failed(ll_kv_attention(rq.data_ptr(), S, H, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 6.f, 256.f, wk.data_ptr(),
                             wv.data_ptr(), keys, scale, out.data_ptr(), stream),
             "ll_kv_attention"))
    return nullptr;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// cache_write(k, v, first token, tokens, rule, (values, scales, amax) of the K slot, of the V slot, k_sink, v_sink) -> True, or
// None when it does not take the call.  The sinks: (parts, epoch) that the producers of k and v were given, or None for both.
PyObject* py_cache_write(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9 || !plain(args[0])) Py_RETURN_NONE;
  const int dev = current_device_of(THPVariable_Unpack(args[0]));
  if (dev < 0) Py_RETURN_NONE;
  const Tensor *k = as_chunk(args[0], dev), *v = as_chunk(args[1], dev);
  const int64_t first = PyLong_AsLongLong(args[2]), tokens = PyLong_AsLongLong(args[3]);
  const int rule = (int)PyLong_AsLong(args[4]);
  if (PyErr_Occurred()) return nullptr;
  if (!k || !v || k->sizes() != v->sizes() || first < 0 || tokens <= 0 || first + tokens > k->size(1)) Py_RETURN_NONE;
  const int64_t M = tokens * k->size(2), Mp = round_up(M, 128);
  uint8_t* out[2][2];
  float* amax[2];
  for (int i = 0; i < 2; ++i) {
    PyObject* t = args[5 + i];
    if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != 3) Py_RETURN_NONE;
    const Tensor *values = as_tensor(PyTuple_GET_ITEM(t, 0)), *scales = as_tensor(PyTuple_GET_ITEM(t, 1)),
        *a = as_tensor(PyTuple_GET_ITEM(t, 2));
    if (!values || !scales || !a || !on_device(*values, dev) || !on_device(*scales, dev) || !on_device(*a, dev) ||
        values->scalar_type() != at::kByte || values->dim() != 2 || values->size(0) != Mp || values->size(1) != 64 ||
        scales->numel() != Mp * 8 || scales->element_size() != 1 || a->numel() != 1 || a->scalar_type() != at::kFloat ||
        !values->is_contiguous() || !scales->is_contiguous())
      Py_RETURN_NONE;
    out[i][0] = values->data_ptr<uint8_t>();
    out[i][1] = static_cast<uint8_t*>(scales->data_ptr());
    amax[i] = a->data_ptr<float>();
  }
  if (out[0][0] == out[1][0] || out[0][1] == out[1][1] || amax[0] == amax[1]) Py_RETURN_NONE;
  const int64_t at = first * k->size(2) * 128;
  const uint16_t *kx = static_cast<const uint16_t*>(k->data_ptr()) + at, *vx = static_cast<const uint16_t*>(v->data_ptr()) + at;
  void* stream = stream_of(dev);
  int code;
  if (args[7] != Py_None || args[8] != Py_None) {
    ll_amax_sink sinks[2];
    if (!parse_sink(args[7], dev, sinks[0]) || !parse_sink(args[8], dev, sinks[1]) || sinks[0].parts == sinks[1].parts) {
      if (PyErr_Occurred()) return nullptr;
      Py_RETURN_NONE;
    }
    code = ll_nvfp4_quantize_pair_from_sinks(kx, vx, M, 128, 128, rule, out[0][0], out[1][0], out[0][1], out[1][1], amax[0],
                                             amax[1], &sinks[0], &sinks[1], stream);
  } else {
    code = LL_ENOSUP;
    if (one_pass_tiles(M, 128, 2)) {
      Epochs e = epochs_of_stream(dev, stream);
      if (e.parts) {
        const ll_amax_sink sink = e.take();
        code = ll_nvfp4_quantize_one_pass(kx, vx, M, 128, 128, rule, out[0][0], out[1][0], out[0][1], out[1][1], amax[0], amax[1], &sink,
                                          LL_EXCHANGE_LOOKS, stream);
      }
    }
    if (code == LL_ENOSUP) {
      const Tensor ws = empty({2 * (int64_t)LL_AMAX_PARTS}, at::kFloat, dev);
      code = ll_nvfp4_quantize_pair(kx, vx, M, 128, 128, rule, out[0][0], out[1][0], out[0][1], out[1][1], amax[0], amax[1],
                                    ws.data_ptr<float>(), stream);
    }
  }
  if (failed(code, "cache write")) return nullptr;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// Calls that took torch's own operations before stay with them where Python code or torch itself has to see each one, or
// where a gradient is wanted.
inline bool traced() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
         torch::jit::tracer::isTracing() || at::autocast::is_autocast_enabled(c10::kCUDA);
}
inline bool needs_torch(const Tensor& t) {
  // batched and functional wrappers have no storage
  return !t.has_storage() || (t.requires_grad() && c10::GradMode::is_enabled()) ||
         (torch::autograd::impl::get_autograd_meta(t) && t._fw_grad(0).defined());
}
// A bf16 matrix [rows, cols] (or, rows < 0, a vector [cols]) on the device, contiguous and 16-byte aligned; null if it is not.
inline const Tensor* as_weight(PyObject* o, int dev, int64_t rows, int64_t cols) {
  if (!plain(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (needs_torch(t) || !is_bf16(t, dev) || !t.is_contiguous() || t.numel() != (rows < 0 ? cols : rows * cols) ||
      !aligned16(t.data_ptr()))
    return nullptr;
  return &t;
}

// The ends of the model: calls of up to kPatchTokens tokens are taken here, larger ones are left to the Python path.  us, kernels of
// patch_linear.hip / torch's matrix product and permuted copy, on the GPU alone:
//                   embedding, tokens                          head without its normalization
//       width       368          720          1012             368          720          1012
//       512         8.9 / 8.6    9.1 / 8.8    9.1 / 8.7        9.1 / 9.2    9.2 / 9.6    9.2 / 9.9
//       1536        9.1 / 9.3    10.7 / 10.6  10.9 / 10.7      14.5 / 9.8   14.6 / 10.5  14.6 / 10.8
//       2304        9.2 / 9.3    11.0 / 10.5  14.8 / 12.3      19.5 / 10.2  19.7 / 11.7  19.7 / 12.0
//       3072        10.8 / 10.8  14.3 / 12.4  14.9 / 13.0      22.1 / 11.0  22.3 / 12.6  22.0 / 13.1
// and on the host: embedding 7 / 30 (35 in Python), head 21 / 43 (75).  The embedding comes first in a forward: where the GPU has
// waited for the host (at every chunk, whose time steps are read back) its host time is all waited for, so the kernel takes every
// call.  The head comes last: its host time matters only while the blocks, whose products grow with tokens x width^2, keep the
// GPU less busy than the host.  A forward of two layers, us, head by the kernel / in Python, with tokens x width^2 in 10^9: 1024 x
// 896 (0.94) 529 / 552, 1536 x 384 (0.91) 496 / 539, 2304 x 192 (1.0) 555 / 562, 1536 x 768 (1.8) 632 / 635, 3072 x 192 (1.8)
// 610 / 607, 2304 x 384 (2.0) 614 / 614, 3072 x 384 (3.6) 764 / 752, 2304 x 768 (4.1) 774 / 767.  Beyond the line the head runs
// on torch's operations, the same bits as in Python, without Python between them.
constexpr int64_t kPatchTokens = 1024;
inline bool head_kernel_takes(int64_t tokens, int64_t width) { return tokens * width * width <= 3ll << 29; }

// patch_embed(x [C, F, H, W], weight, bias or None, outputs, pt, ph, pw) -> tokens [1, f h w, outputs], or None when it does not
// take the call.
PyObject* py_patch_embed(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7 || !plain(args[0]) || traced()) Py_RETURN_NONE;
  const Tensor& x = THPVariable_Unpack(args[0]);
  const int dev = current_device_of(x);
  if (needs_torch(x) || !is_bf16(x, dev) || x.dim() != 4 || !x.is_contiguous() || x.numel() == 0 || x.numel() >= (1ll << 31))
    Py_RETURN_NONE;
  const int64_t N = PyLong_AsLongLong(args[3]), pt = PyLong_AsLongLong(args[4]), ph = PyLong_AsLongLong(args[5]),
      pw = PyLong_AsLongLong(args[6]);
  if (PyErr_Occurred()) return nullptr;
  if (pt < 1 || ph < 1 || pw < 1 || x.size(1) < pt || x.size(2) < ph || x.size(3) < pw || N < 1 || N > (1 << 20)) Py_RETURN_NONE;
  const int64_t f = x.size(1) / pt, h = x.size(2) / ph, wd = x.size(3) / pw;
  if (f * h * wd > kPatchTokens) Py_RETURN_NONE;
  const Tensor* w = as_weight(args[1], dev, N, x.size(0) * pt * ph * pw);
  const Tensor* b = args[2] == Py_None ? nullptr : as_weight(args[2], dev, -1, N);
  if (!w || (!b && args[2] != Py_None)) Py_RETURN_NONE;
  const Tensor out = empty({1, f * h * wd, N}, at::kBFloat16, dev);
  const int code = ll_patch_embed(x.data_ptr(), (int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3), (int)pt,
                                  (int)ph, (int)pw, w->data_ptr(), b ? b->data_ptr() : nullptr, (int)N, out.data_ptr(),
                                  stream_of(dev));
  if (code == LL_ENOSUP) Py_RETURN_NONE;
  if (failed(code, "ll_patch_embed")) return nullptr;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// head(x [1, L, C], e [1, F, 2, C] (shift, scale), weight, bias or None, eps, channels, (f, h, w), (pt, ph, pw)) -> latents
// [channels, f pt, h ph, w pw], or None when it does not take the call: LayerNorm(x) * (1 + scale) + shift, linear layer, unpatchify.
PyObject* py_head(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 || !plain(args[0]) || !plain(args[1]) || traced()) Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(args[0]), &e = THPVariable_Unpack(args[1]);
  const int dev = current_device_of(x);
  if (needs_torch(x) || needs_torch(e) || !is_bf16(x, dev) || !is_bf16(e, dev) || x.dim() != 3 || x.size(0) != 1 ||
      !x.is_contiguous() || e.dim() != 4 || e.size(0) != 1 || e.size(2) != 2 || e.size(3) != x.size(2) || !e.is_contiguous() ||
      x.numel() == 0)
    Py_RETURN_NONE;
  const int64_t L = x.size(1), C = x.size(2), F = e.size(1);
  int64_t grid[3], patch[3];
  for (int i = 0; i < 2; ++i) {
    PyObject* t = args[6 + i];
    if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != 3) Py_RETURN_NONE;
    for (int j = 0; j < 3; ++j) (i ? patch : grid)[j] = PyLong_AsLongLong(PyTuple_GET_ITEM(t, j));
  }
  const double eps = PyFloat_AsDouble(args[4]);
  const int64_t channels = PyLong_AsLongLong(args[5]);
  if (PyErr_Occurred()) return nullptr;
  for (int j = 0; j < 3; ++j)
    if (grid[j] < 1 || patch[j] < 1) Py_RETURN_NONE;
  if (F < 1 || L % F || L > kPatchTokens || grid[0] * grid[1] * grid[2] != L || C % 16 || channels < 1 ||
      !aligned16(x.data_ptr()) || !aligned16(e.data_ptr()))
    Py_RETURN_NONE;
  const int64_t N = channels * patch[0] * patch[1] * patch[2];
  if (N >= (1 << 20) || N * L >= (1ll << 31)) Py_RETURN_NONE;
  const Tensor* w = as_weight(args[2], dev, N, C);
  const Tensor* b = args[3] == Py_None ? nullptr : as_weight(args[3], dev, -1, N);
  if (!w || (!b && args[3] != Py_None)) Py_RETURN_NONE;
  void* stream = stream_of(dev);
  const Tensor y = empty({L, C}, at::kBFloat16, dev);
  const uint16_t* shift = static_cast<const uint16_t*>(e.data_ptr());
  if (failed(ll_adaln_modulate_amax(x.data_ptr(), 1, L, (int)C, shift + C, shift, e.stride(0), e.stride(1), e.stride(0),
                                    e.stride(1), L / F, (float)eps, 1, y.data_ptr(), nullptr, stream), "ll_adaln_modulate"))
    return nullptr;
  const int64_t extent[4] = {channels, grid[0] * patch[0], grid[1] * patch[1], grid[2] * patch[2]};
  if (!head_kernel_takes(L, C)) {
    at::AutoDispatchBelowADInplaceOrView no_autograd;
    const Tensor rows = at::linear(y, *w, b ? std::optional<Tensor>(*b) : std::nullopt);
    return THPVariable_Wrap(rows.view({grid[0], grid[1], grid[2], patch[0], patch[1], patch[2], channels})
                                .permute({6, 0, 3, 1, 4, 2, 5}).reshape(extent));
  }
  const Tensor out = empty(extent, at::kBFloat16, dev);
  if (failed(ll_patch_head(y.data_ptr(), (int)C, w->data_ptr(), b ? b->data_ptr() : nullptr, (int)channels, (int)out.size(1),
                           (int)out.size(2), (int)out.size(3), (int)patch[0], (int)patch[1], (int)patch[2], out.data_ptr(),
                           stream), "ll_patch_head"))
    return nullptr;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// unipc_step(flow, sample, last or None, m1 or None, m2 or None, sigma, corrector, predictor) -> (x0 prediction, corrected
// sample, next sample), or None when it does not take the call.  corrector, predictor: (order, ratio, m0, b, rho, rk,
// rho_new), see ll_unipc_scalars; with a corrector of order 0 the corrected sample is `sample` itself.
PyObject* py_unipc_step(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 || traced()) Py_RETURN_NONE;
  const Tensor* in[5] = {};
  int dev = -1;
  for (int i = 0; i < 5; ++i) {
    if (i > 1 && args[i] == Py_None) continue;
    if (!plain(args[i])) Py_RETURN_NONE;
    const Tensor& t = THPVariable_Unpack(args[i]);
    if (needs_torch(t)) Py_RETURN_NONE;
    if (i == 0) dev = current_device_of(t);
    if (!is_bf16(t, dev) || !t.is_contiguous() || t.numel() == 0 || (i > 0 && t.sizes() != in[0]->sizes())) Py_RETURN_NONE;
    in[i] = &t;
  }
  const double sigma = PyFloat_AsDouble(args[5]);
  ll_unipc_scalars s[2];
  for (int i = 0; i < 2; ++i) {
    PyObject* t = args[6 + i];
    if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != 7) Py_RETURN_NONE;
    s[i].order = (int)PyLong_AsLong(PyTuple_GET_ITEM(t, 0));
    float* const f[6] = {&s[i].ratio, &s[i].m0, &s[i].b, &s[i].rho, &s[i].rk, &s[i].rho_new};
    for (int j = 0; j < 6; ++j) *f[j] = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(t, 1 + j));
  }
  if (PyErr_Occurred()) return nullptr;
  const bool correct = s[0].order > 0;
  const Tensor converted = empty(in[0]->sizes(), at::kBFloat16, dev), next = empty(in[0]->sizes(), at::kBFloat16, dev);
  const Tensor corrected = correct ? empty(in[0]->sizes(), at::kBFloat16, dev) : *in[1];
  const auto ptr = [&](int i) -> const void* { return in[i] ? in[i]->data_ptr() : nullptr; };
  if (failed(ll_unipc_step(ptr(0), ptr(1), ptr(2), ptr(3), ptr(4), in[0]->numel(), (float)sigma, &s[0], &s[1], converted.data_ptr(),
                           correct ? corrected.data_ptr() : nullptr, next.data_ptr(), stream_of(dev)),
             "ll_unipc_step"))
    return nullptr;
  return tuple3(converted, corrected, next);
  END_HANDLE_TH_ERRORS
}

// recording(device index, -1: the current one) -> whether launches on the device's current stream are being recorded
PyObject* py_recording(PyObject*, PyObject* arg) {
  HANDLE_TH_ERRORS
  const int64_t dev = PyLong_AsLongLong(arg);
  if (PyErr_Occurred()) return nullptr;
  if (recording(stream_of(dev < 0 ? c10::hip::current_device() : (int)dev))) Py_RETURN_TRUE;
  Py_RETURN_FALSE;
  END_HANDLE_TH_ERRORS
}

// current_stream() -> the current HIP stream of the current device as an integer
PyObject* py_current_stream(PyObject*, PyObject*) {
  HANDLE_TH_ERRORS
  return PyLong_FromVoidPtr(stream_of(c10::hip::current_device()));
  END_HANDLE_TH_ERRORS
}

// release_stream_sink(): gives back the amax sink of (current device, current stream)
PyObject* py_release_stream_sink(PyObject*, PyObject*) {
  HANDLE_TH_ERRORS
  const int dev = c10::hip::current_device();
  std::lock_guard<std::mutex> lock(g_sink_mutex);
  stream_sinks().erase({dev, stream_of(dev)});
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"block_forward", (PyCFunction)(void (*)(void))py_block_forward, METH_FASTCALL, nullptr},
    {"slot_addresses", (PyCFunction)(void (*)(void))py_slot_addresses, METH_FASTCALL, nullptr},
    {"kv_attention", (PyCFunction)(void (*)(void))py_kv_attention, METH_FASTCALL, nullptr},
    {"kv_attention_relative", (PyCFunction)(void (*)(void))py_kv_attention_relative, METH_FASTCALL, nullptr},
    {"cache_write", (PyCFunction)(void (*)(void))py_cache_write, METH_FASTCALL, nullptr},
    {"patch_embed", (PyCFunction)(void (*)(void))py_patch_embed, METH_FASTCALL, nullptr},
    {"head", (PyCFunction)(void (*)(void))py_head, METH_FASTCALL, nullptr},
    {"unipc_step", (PyCFunction)(void (*)(void))py_unipc_step, METH_FASTCALL, nullptr},
    {"recording", py_recording, METH_O, nullptr},
    {"current_stream", py_current_stream, METH_NOARGS, nullptr},
    {"release_stream_sink", py_release_stream_sink, METH_NOARGS, nullptr},
    {"quantize", (PyCFunction)(void (*)(void))py_quantize, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))py_linear, METH_FASTCALL, nullptr},
    {"dequantize", (PyCFunction)(void (*)(void))py_dequantize, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_ops(void) {
  PyObject* m = PyModule_Create(&module);
  if (m) PyModule_AddIntConstant(m, "EPOCHS_PER_CALL", kEpochsPerCall);
  if (m) PyModule_AddIntConstant(m, "PATCH_TOKENS", kPatchTokens);
  if (m) PyModule_AddStringConstant(m, "TORCH_VERSION", LL_TORCH_VERSION);
  return m;
}
