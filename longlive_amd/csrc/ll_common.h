// Shared device/host helpers for the gfx950 NVFP4 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <atomic>

#include "../../include/ll_nvfp4.h"
#include "scratch_sets.h"

namespace ll {

// ----------------------------------------------------------------------------- errors
void set_error(const char* fmt, ...);

#define LL_REQUIRE(cond, ...)      \
  do {                             \
    if (!(cond)) {                 \
      ll::set_error(__VA_ARGS__);  \
      return LL_EINVAL;            \
    }                              \
  } while (0)

#define LL_CHECK_LAUNCH(name)                                              \
  do {                                                                     \
    hipError_t e__ = hipGetLastError();                                    \
    if (e__ != hipSuccess) {                                               \
      ll::set_error("%s: launch failed: %s", name, hipGetErrorString(e__)); \
      return LL_ELAUNCH;                                                   \
    }                                                                      \
  } while (0)

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// ----------------------------------------------------------------------------- memory of the library's own (stream_scratch.hip)
// A set with at least record_bytes and `counters` counters (scratch_sets.h).  may_allocate false (the stream is being
// captured into a graph): only a set that is already large enough is handed out, and *missing says that there is none.
int stream_scratch(int dev, hipStream_t stream, size_t record_bytes, size_t counters, bool may_allocate, StreamScratch& out,
                   bool* missing, const char* what);
// The records and counters of the small products of a stream; false where there is none to be had (the stream is being
// captured, the allocation fails): no error, the launch then takes its way without memory.
bool small_product_scratch(int dev, hipStream_t stream, int cus, StreamScratch& out);
int release_stream_scratch(int dev, hipStream_t stream);
// Whether work submitted to `stream` is being recorded into a graph instead of run.  A failing query (the legacy
// stream while another stream of the thread captures) counts as recording: then nothing may be allocated either.
bool stream_is_capturing(hipStream_t stream);
int compute_units_of(int dev, int& cus, const char* what);

// Kernels that need more than 64 KB of dynamic LDS have to be told so with hipFuncSetAttribute, and that setting
// holds per device.  `done` (one per kernel, zero-initialised) keeps one bit per device ordinal so that the call
// is made once for every device the kernel is launched on; two threads racing here both make the same call.
inline int allow_dynamic_lds(const void* kernel, size_t bytes, std::atomic<uint64_t>& done, const char* what) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error("%s: hipGetDevice failed: %s", what, hipGetErrorString(e));
    return LL_ELAUNCH;
  }
  const uint64_t bit = 1ull << (dev & 63);
  if (dev < 64 && (done.load(std::memory_order_acquire) & bit)) return LL_OK;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e != hipSuccess) {
    set_error("%s: cannot reserve %zu bytes of LDS: %s", what, bytes, hipGetErrorString(e));
    return LL_ELAUNCH;
  }
  if (dev < 64) done.fetch_or(bit, std::memory_order_release);
  return LL_OK;
}

// ----------------------------------------------------------------------------- formats
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }

// fp32 -> bf16 bits, round to nearest even, with the hardware conversion of gfx950 (v_cvt_pk_bf16_f32;
// NaN becomes a quiet NaN).
typedef __bf16 bf16x2_hw __attribute__((ext_vector_type(2)));
typedef float f32x2_hw __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  return (uint32_t)__builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}
// Two values at once: lo in bits 0-15, hi in bits 16-31.
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const f32x2_hw v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_hw));
}
// Two at once: one conversion for both.
__device__ __forceinline__ void round_to_bf16(float& a, float& b) {
  const uint32_t w = pack_bf16x2(a, b);
  a = __uint_as_float(w << 16);
  b = __uint_as_float(w & 0xFFFF0000u);
}
__device__ __forceinline__ float round_to_bf16(float f) { return __uint_as_float(f32_to_bf16_bits(f) << 16); }

// e4m3fn byte -> fp32 (exact). 0x7F / 0xFF decode to NaN.
__device__ __forceinline__ float e4m3_to_f32(uint32_t b) {
  uint32_t e = (b >> 3) & 0xFu, m = b & 7u;
  float v;
  if (e == 0) {
    v = (float)m * 0.001953125f;  // m * 2^-9
  } else if (e == 15 && m == 7) {
    v = __uint_as_float(0x7FC00000u);
  } else {
    v = __uint_as_float(((e + 120u) << 23) | (m << 20));
  }
  return (b & 0x80u) ? -v : v;
}

typedef float float2v __attribute__((ext_vector_type(2)));
// The eight e2m1 values of one packed dword, exact, in four conversions.
__device__ __forceinline__ void fp4x8_values(uint32_t w, float (&q)[8]) {
  const float2v p0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 0);
  const float2v p1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 1);
  const float2v p2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 2);
  const float2v p3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 3);
  q[0] = p0[0]; q[1] = p0[1]; q[2] = p1[0]; q[3] = p1[1];
  q[4] = p2[0]; q[5] = p2[1]; q[6] = p3[0]; q[7] = p3[1];
}

// fp32 -> e4m3fn byte, round to nearest even, |x| > 464 -> NaN (0x7F): the value torch's
// float8_e4m3fn cast produces.
__device__ __forceinline__ uint32_t f32_to_e4m3(float x) {
  uint32_t u = __float_as_uint(x);
  uint32_t sign = (u >> 24) & 0x80u;
  u &= 0x7FFFFFFFu;
  float a = __uint_as_float(u);
  if (!(a <= 464.0f)) return sign | 0x7Fu;  // NaN, inf, overflow
  if (a >= 0.015625f) {                     // normal range: keep 3 mantissa bits
    uint32_t r = (u + 0x7FFFFu + ((u >> 20) & 1u)) >> 20;
    return sign | (r - (120u << 3));
  }
  return sign | (uint32_t)__builtin_rintf(a * 512.0f);  // sub-normal grid 2^-9, 8 -> 2^-6
}

// Offset of scale (r, c) of a [rows, cols] e4m3 matrix stored in 128x4 blocked order.
__host__ __device__ __forceinline__ int64_t blocked_scale_offset(int64_t r, int64_t c, int64_t cols) {
  int64_t rb = r >> 7, ri = r & 127, cb = c >> 2, ci = c & 3;
  return ((rb * (cols >> 2) + cb) * 32 + (ri & 31)) * 16 + (ri >> 5) * 4 + ci;
}

__host__ __device__ __forceinline__ void rule_limits(int rule, float& e2, float& e4) {
  e2 = (rule == LL_RULE_STATIC_4) ? 4.0f : 6.0f;
  e4 = (rule == LL_RULE_STATIC_6 || rule == LL_RULE_STATIC_4) ? 448.0f : 256.0f;
}

// 1 / (e2m1_max * e4m3_max) of a KV-cache slot as the reference's fused dequantization forms it: the reciprocal
// in double, rounded to fp32 once (utils/kernel/kv_dequant_cuda.cu:216); the slot scale is amax times this.
inline float kv_inverse_denominator(float e2m1_max, float e4m3_max) {
  return static_cast<float>(1.0 / (static_cast<double>(e2m1_max) * static_cast<double>(e4m3_max)));
}

// ----------------------------------------------------------------------------- wave helpers
// Maxima by data-parallel-primitive moves instead of LDS permutes, which are a trip to LDS each, one behind the other.  A lane
// that a move does not reach keeps its own value.  All 64 lanes are active.
#define LL_DPP_MAX(v, ctrl, row_mask)                                                                                \
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), ctrl, row_mask, 0xF, false)))
// Over 16 neighbouring lanes, in every one of them; see sum_over_16_lanes.
__device__ __forceinline__ float max_over_16_lanes(float v) {
  LL_DPP_MAX(v, 0xB1, 0xF);   // quad_perm [1, 0, 3, 2]
  LL_DPP_MAX(v, 0x4E, 0xF);   // quad_perm [2, 3, 0, 1]
  LL_DPP_MAX(v, 0x141, 0xF);  // row_half_mirror
  LL_DPP_MAX(v, 0x140, 0xF);  // row_mirror
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  v = max_over_16_lanes(v);
  LL_DPP_MAX(v, 0x142, 0xA);  // row_bcast:15 into rows 1 and 3
  LL_DPP_MAX(v, 0x143, 0xC);  // row_bcast:31 into rows 2 and 3
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
#undef LL_DPP_MAX
// Sum over the wave with data-parallel-primitive moves instead of LDS permutes: partial sums travel down
// each row of 16 lanes (row_shr 1, 2, 3, then 4 and 8 under bank masks), then across the rows (row_bcast 15
// and 31), which leaves the total in lane 63; every lane returns that value.  Lanes that a move does not
// reach contribute 0 (bound_ctrl).
#define LL_DPP_ADD(v, ctrl, row_mask, bank_mask)                                                                 \
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, row_mask, bank_mask, true))
__device__ __forceinline__ float wave_sum_dpp(float v) {
  LL_DPP_ADD(v, 0x111, 0xF, 0xF);  // row_shr:1
  LL_DPP_ADD(v, 0x112, 0xF, 0xF);  // row_shr:2
  LL_DPP_ADD(v, 0x114, 0xF, 0xE);  // row_shr:4, lanes 4-15 of each row
  LL_DPP_ADD(v, 0x118, 0xF, 0xC);  // row_shr:8, lanes 8-15 of each row
  LL_DPP_ADD(v, 0x142, 0xA, 0xF);  // row_bcast:15 into rows 1 and 3
  LL_DPP_ADD(v, 0x143, 0xC, 0xF);  // row_bcast:31 into rows 2 and 3
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
// The same over each half of the wave, in all lanes of it: the bits that wave_sum_dpp has for 32 values and zeros behind them.
__device__ __forceinline__ float half_wave_sum_dpp(float v) {
  LL_DPP_ADD(v, 0x111, 0xF, 0xF);
  LL_DPP_ADD(v, 0x112, 0xF, 0xF);
  LL_DPP_ADD(v, 0x114, 0xF, 0xE);
  LL_DPP_ADD(v, 0x118, 0xF, 0xC);
  LL_DPP_ADD(v, 0x142, 0xA, 0xF);
  const int lower = __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 31), upper = __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63);
  return __builtin_bit_cast(float, (threadIdx.x & 32) ? upper : lower);
}
// Sum over 16 neighbouring lanes, in every one of them: over lanes 1, 2, 4 and 8 apart in turn.  (When the lanes of a quad agree, the
// mirrored lane of the other quad stands for the one 4 apart, and likewise for 8.)
__device__ __forceinline__ float sum_over_16_lanes(float v) {
  LL_DPP_ADD(v, 0xB1, 0xF, 0xF);   // quad_perm [1, 0, 3, 2]
  LL_DPP_ADD(v, 0x4E, 0xF, 0xF);   // quad_perm [2, 3, 0, 1]
  LL_DPP_ADD(v, 0x141, 0xF, 0xF);  // row_half_mirror
  LL_DPP_ADD(v, 0x140, 0xF, 0xF);  // row_mirror
  return v;
}
#undef LL_DPP_ADD

// n / d for any 32-bit n in five instructions (Granlund and Montgomery, Division by invariant integers using multiplication).
struct Divisor {
  uint32_t d, m, s1, s2;
};
inline Divisor divisor(uint32_t d) {
  uint32_t l = 0;
  while (l < 32 && (1ull << l) < d) ++l;
  return Divisor{d, (uint32_t)(((1ull << 32) * ((1ull << l) - d)) / d + 1), l < 1 ? l : 1, l > 1 ? l - 1 : 0};
}
__device__ __forceinline__ uint32_t operator/(uint32_t n, const Divisor& by) {
  const uint32_t t = __umulhi(by.m, n);
  return (t + ((n - t) >> by.s1)) >> by.s2;
}

// Load through a pointer that is known to address global memory.  Slot pointers come out of a table, so
// the compiler would otherwise emit flat loads, whose completion also counts as an LDS event and stalls
// the first LDS wait that follows.
template <typename T>
__device__ __forceinline__ T load_global(const void* ptr) {
  return *(const __attribute__((address_space(1))) T*)ptr;
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// One store of 16 bytes.  Left to itself the compiler merges the ends of a kernel's branches and stores 12 and 4, or 4 and 12.
__device__ __forceinline__ void store_b128(void* dst, u32x4 v) {
  asm volatile("" : "+v"(v));
  *reinterpret_cast<u32x4*>(dst) = v;
}

// max(m, |v|) over the 8 bf16 values of a packed 16-byte group
__device__ __forceinline__ float abs_max_bf16x8(const uint4& v, float m) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m = fmaxf(m, fabsf(__uint_as_float(w[i] << 16)));
    m = fmaxf(m, fabsf(__uint_as_float(w[i] & 0xFFFF0000u)));
  }
  return m;
}
// Amax sink: a kernel that writes a tensor leaves partial absolute maxima of it in LL_AMAX_PARTS 64-bit
// slots, each holding (epoch << 32) | float bits and raised with a 64-bit atomic max.  A value of a newer
// epoch beats every older one, so the slots never need clearing; the reader ignores slots of other epochs.
// (The bit patterns of non-negative floats order like unsigned integers.)
constexpr int kAmaxParts = LL_AMAX_PARTS;
struct AmaxSink {
  unsigned long long* parts;     // null: no sink
  uint32_t epoch;
  const uint32_t* epoch_offset;  // device word added to epoch when the kernel runs (launches replayed from a graph), or null
};
__device__ __forceinline__ uint32_t amax_sink_epoch(uint32_t epoch, const uint32_t* epoch_offset) {
  return epoch + (epoch_offset ? *epoch_offset : 0u);
}
__device__ __forceinline__ void amax_sink_update(const AmaxSink& sink, uint32_t slot, float v) {
  const uint32_t epoch = amax_sink_epoch(sink.epoch, sink.epoch_offset);
  atomicMax(sink.parts + (slot & (kAmaxParts - 1)), ((unsigned long long)epoch << 32) | __float_as_uint(v));
}
// The kernel-side sink of a caller's ll_amax_sink (null or without a buffer: no sink).
inline AmaxSink make_sink(const ll_amax_sink* s) {
  AmaxSink k{};
  if (s && s->parts) {
    k.parts = reinterpret_cast<unsigned long long*>(s->parts);
    k.epoch = s->epoch;
    k.epoch_offset = s->epoch_offset;
  }
  return k;
}
inline bool sink_is_valid(const ll_amax_sink* s) {
  return !s || !s->parts ||
         ((reinterpret_cast<uintptr_t>(s->parts) & 7) == 0 && s->epoch != 0 && (reinterpret_cast<uintptr_t>(s->epoch_offset) & 3) == 0);
}
__device__ __forceinline__ float amax_sink_read(const unsigned long long* parts, uint32_t epoch, int slot) {
  const unsigned long long v = parts[slot];
  return (uint32_t)(v >> 32) == epoch ? __uint_as_float((uint32_t)v) : 0.0f;
}

}  // namespace ll
