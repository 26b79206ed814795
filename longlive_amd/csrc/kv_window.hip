// The chunk's side of attention over the KV cache for gfx950, everything that comes before the attention kernel itself:
//
//  * ll_kv_smooth        k - mean(k over the head dimension) (utils/quant.py:797-798), mean and difference rounded to bf16 as
//                        the two eager operations round them
//  * ll_kv_window_rope   relative RoPE (wan_5b/modules/causal_model.py:486-487, 716-771): the attended window as bf16 K
//                        and V, [cached slots | chunk], K rotated by the window's own positions, and the rotated queries
//
// Both are bound by the latency of memory and, for large windows, by its bandwidth: 368 queries x 16 heads over 1104 cached + 368
// keys, 21 MB, 5.4 us, 2640 x 24 over 10560 + 2640, 260 MB, 60 us.  (6.3 and 63 with flat loads from the slots, the angles loaded behind
// them, and stores split in two.)  As separate operations (pointer tables copied to the device, two dequantizations, mean,
// difference, two concatenations, two rotations) the window moved every byte four times in 13 launches and synchronised
// the host for the tables: 368 tokens of 16 heads behind 1104 cached ones took 230 us, 62 us of them on the GPU.  Here each
// value is read once and written once; a workgroup's 256 threads hold 16 (token, head) rows, 16 lanes a row, so that the
// mean over a head needs only moves between the lanes of a row.
#include "ll_common.h"
#include "norm_rows.h"

#pragma clang fp contract(off)

namespace ll {

// The sum over the 16 lanes that hold a head, in the order of qk_norm_rope_kernel.  torch's mean adds in another order: where a
// mean lies at the edge between two bf16 values the two may round apart (none of 8 million values drawn from N(0, 1) did).
__device__ __forceinline__ float head_sum(float v) { return sum_over_16_lanes(v); }

// v - mean(v) of a head, with the roundings of the two eager bf16 operations.
__device__ __forceinline__ void smooth8(float (&v)[8]) {
  float part = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) part += v[j];
  const float mean = round_to_bf16(head_sum(part) * (1.0f / 128.0f));
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = round_to_bf16(v[j] - mean);
}

__device__ __forceinline__ void rotate8(float (&v)[8], const float4& cs, const float4& sn) {
  const float cc[4] = {cs.x, cs.y, cs.z, cs.w}, ss[4] = {sn.x, sn.y, sn.z, sn.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = v[2 * i], b = v[2 * i + 1];
    v[2 * i] = a * cc[i] - b * ss[i];
    v[2 * i + 1] = a * ss[i] + b * cc[i];
  }
}

constexpr int kRowsPerWindowWg = 16;  // (token, head) rows of 16 lanes

__global__ __launch_bounds__(256) void kv_smooth_kernel(const uint16_t* __restrict__ k, uint32_t rows, uint16_t* __restrict__ out) {
  const uint32_t row = blockIdx.x * kRowsPerWindowWg + (threadIdx.x >> 4);
  if (row >= rows) return;  // uniform over the 16 lanes of a row
  const int64_t at = (int64_t)row * 128 + (threadIdx.x & 15) * 8;
  float v[8];
  unpack8(*reinterpret_cast<const uint4*>(k + at), v);
  smooth8(v);
  *reinterpret_cast<uint4*>(out + at) = pack8(v);
}

struct WindowSide {  // K or V of the window
  const uint64_t *values, *scales, *amax;  // slot pointers
  const uint16_t* fresh;                   // the chunk's, [n_new, H, 128]
  uint16_t* out;                           // [n_cached + n_new, H, 128]
};
struct WindowParams {
  WindowSide k, v;
  const uint16_t* q;
  uint16_t* q_out;
  const float *cos_k, *sin_k, *cos_q, *sin_q;  // rows of 64: one per key, one per query
  Divisor H, slot_tokens;
  uint32_t Lq, n_cached, n_new;
  float inv_denom;
  uint32_t wgs_window, wgs_q;  // workgroups of one side of the window, of the queries
};

// Workgroups [0, wgs_window): K, then wgs_window for V, then wgs_q for the queries.  Windows of a few thousand tokens are bound by
// the chain (slot pointers, bytes, store) and by the instructions of a thread, about 200 for its eight values: a division is a
// product and a scale byte one conversion.  us, with divisions and the scale taken apart / so: 368 queries x 16 heads over 1104 +
// 368 keys 5.8 / 5.4, 880 x 12 over 3520 + 880 10.9 / 10.4, 2640 x 24 over 10560 + 2640 61.7 / 60.  Two rows a thread, their loads
// under way together: 6.0, 11.4 and 57.9, but 2.6 instead of 2.15 for 64 x 2 over 128 + 64.
__global__ __launch_bounds__(256) void kv_window_rope_kernel(WindowParams p) {
  const int c = (threadIdx.x & 15) * 8;  // element of the head
  uint32_t wg = blockIdx.x;
  if (wg >= 2 * p.wgs_window) {
    const uint32_t row = (wg - 2 * p.wgs_window) * kRowsPerWindowWg + (threadIdx.x >> 4);
    if (row >= p.Lq * p.H.d) return;
    const int64_t angles = (int64_t)(row / p.H) * 64 + (c >> 1);
    float v[8];
    unpack8(*reinterpret_cast<const uint4*>(p.q + (int64_t)row * 128 + c), v);
    rotate8(v, *reinterpret_cast<const float4*>(p.cos_q + angles), *reinterpret_cast<const float4*>(p.sin_q + angles));
    store_b128(p.q_out + (int64_t)row * 128 + c, __builtin_bit_cast(u32x4, pack8(v)));
    return;
  }
  const bool is_v = wg >= p.wgs_window;
  if (is_v) wg -= p.wgs_window;
  const WindowSide side = is_v ? p.v : p.k;
  const uint32_t cached_rows = p.n_cached * p.H.d, row = wg * kRowsPerWindowWg + (threadIdx.x >> 4);
  if (row >= cached_rows + p.n_new * p.H.d) return;
  const uint32_t t = row / p.H;
  const bool cached = row < cached_rows;
  const uint8_t *values = nullptr, *scales = nullptr, *amax = nullptr;
  uint32_t r = 0;  // row of the slot
  if (cached) {
    const uint32_t slot = t / p.slot_tokens;
    r = row - slot * p.slot_tokens.d * p.H.d;
    values = reinterpret_cast<const uint8_t*>(side.values[slot]);
    scales = reinterpret_cast<const uint8_t*>(side.scales[slot]);
    amax = reinterpret_cast<const uint8_t*>(side.amax[slot]);
  }
  float4 cs{}, sn{};  // on their way while the slot's pointers and then its bytes are
  if (!is_v) {
    cs = *reinterpret_cast<const float4*>(p.cos_k + (int64_t)t * 64 + (c >> 1));
    sn = *reinterpret_cast<const float4*>(p.sin_k + (int64_t)t * 64 + (c >> 1));
  }
  float v[8];
  if (cached) {
    const uint32_t w = load_global<uint32_t>(values + (int64_t)r * 64 + (c >> 1));
    const uint32_t sb = load_global<uint8_t>(scales + blocked_scale_offset(r, c >> 4, 8));
    const float gs = load_global<float>(amax) * p.inv_denom;
    const float s = __builtin_amdgcn_cvt_f32_fp8((int)sb, 0);
    float q[8];
    fp4x8_values(w, q);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (q[j] * s) * gs;  // kv_dequantize_kernel's value, rounded to bf16
#pragma unroll
    for (int j = 0; j < 8; j += 2) round_to_bf16(v[j], v[j + 1]);
  } else {
    unpack8(*reinterpret_cast<const uint4*>(side.fresh + (int64_t)(row - cached_rows) * 128 + c), v);
    if (!is_v) smooth8(v);
  }
  if (!is_v) rotate8(v, cs, sn);
  store_b128(side.out + (int64_t)row * 128 + c, __builtin_bit_cast(u32x4, pack8(v)));
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace ll

extern "C" int ll_kv_smooth(const void* k, int64_t tokens, int num_heads, void* out, void* stream) {
  using namespace ll;
  LL_REQUIRE(k && out && aligned16(k) && aligned16(out), "ll_kv_smooth: pointers must be 16-byte aligned and not null");
  LL_REQUIRE(tokens > 0 && num_heads > 0 && tokens * num_heads <= 0x7FFFFFFF, "ll_kv_smooth: bad shape %lld tokens x %d heads",
             (long long)tokens, num_heads);
  const int64_t rows = tokens * num_heads;
  hipLaunchKernelGGL(kv_smooth_kernel, dim3((unsigned)((rows + kRowsPerWindowWg - 1) / kRowsPerWindowWg)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(k), (uint32_t)rows, static_cast<uint16_t*>(out));
  LL_CHECK_LAUNCH("kv_smooth_kernel");
  return LL_OK;
}

extern "C" int ll_kv_window_rope(const void* q, int64_t Lq, int num_heads, const uint64_t* k_values_ptrs, const uint64_t* k_scales_ptrs,
                                 const uint64_t* k_amax_ptrs, const uint64_t* v_values_ptrs, const uint64_t* v_scales_ptrs,
                                 const uint64_t* v_amax_ptrs, int64_t n_cached, int block_token_size, float e2m1_max, float e4m3_max,
                                 const void* k_new, const void* v_new, int64_t n_new, const float* cos_k, const float* sin_k,
                                 const float* cos_q, const float* sin_q, void* q_out, void* k_out, void* v_out, void* stream) {
  using namespace ll;
  LL_REQUIRE(q && k_new && v_new && cos_k && sin_k && cos_q && sin_q && q_out && k_out && v_out, "ll_kv_window_rope: null pointer");
  LL_REQUIRE(Lq > 0 && n_new > 0 && n_cached >= 0 && num_heads > 0 && (n_cached + n_new) * num_heads <= 0x3FFFFFFF &&
                 Lq * num_heads <= 0x3FFFFFFF,
             "ll_kv_window_rope: bad shape Lq=%lld cached=%lld new=%lld heads=%d", (long long)Lq, (long long)n_cached, (long long)n_new, num_heads);
  LL_REQUIRE(n_cached == 0 || (k_values_ptrs && k_scales_ptrs && k_amax_ptrs && v_values_ptrs && v_scales_ptrs && v_amax_ptrs &&
                               block_token_size > 0 && n_cached % block_token_size == 0),
             "ll_kv_window_rope: cached keys need the slot pointers and whole slots");
  for (const void* ptr : {q, k_new, v_new, (const void*)cos_k, (const void*)sin_k, (const void*)cos_q, (const void*)sin_q,
                          (const void*)q_out, (const void*)k_out, (const void*)v_out})
    LL_REQUIRE(aligned16(ptr), "ll_kv_window_rope: pointers must be 16-byte aligned");
  WindowParams p{};
  p.k = {k_values_ptrs, k_scales_ptrs, k_amax_ptrs, static_cast<const uint16_t*>(k_new), static_cast<uint16_t*>(k_out)};
  p.v = {v_values_ptrs, v_scales_ptrs, v_amax_ptrs, static_cast<const uint16_t*>(v_new), static_cast<uint16_t*>(v_out)};
  p.q = static_cast<const uint16_t*>(q);
  p.q_out = static_cast<uint16_t*>(q_out);
  p.cos_k = cos_k;
  p.sin_k = sin_k;
  p.cos_q = cos_q;
  p.sin_q = sin_q;
  p.H = divisor((uint32_t)num_heads);
  p.Lq = (uint32_t)Lq;
  p.n_cached = (uint32_t)n_cached;
  p.n_new = (uint32_t)n_new;
  p.slot_tokens = divisor(n_cached ? (uint32_t)block_token_size : 1u);
  p.inv_denom = kv_inverse_denominator(e2m1_max, e4m3_max);
  p.wgs_window = (uint32_t)(((n_cached + n_new) * num_heads + kRowsPerWindowWg - 1) / kRowsPerWindowWg);
  p.wgs_q = (uint32_t)((Lq * num_heads + kRowsPerWindowWg - 1) / kRowsPerWindowWg);
  hipLaunchKernelGGL(kv_window_rope_kernel, dim3(2 * p.wgs_window + p.wgs_q), dim3(256), 0, static_cast<hipStream_t>(stream), p);
  LL_CHECK_LAUNCH("kv_window_rope_kernel");
  return LL_OK;
}
