// A W4A4 linear layer of a small activation in one launch: tensor amax, quantization to NVFP4 and the product.
//
// What a product of 48 x 256 x 512 costs is launches and trips to memory: quantization and GEMM are two of either, 4 to 5 us
// each, for a microsecond of work.  Here a workgroup quantizes the 32 rows of its own tile, into LDS, and multiplies them;
// the column tiles of a row quantize it again, which costs nothing while compute units are idle.  The tensor amax comes
// from the sink in which the producer of x left it, or every workgroup forms it from the whole tensor.
//
// Measured, us on the GPU, two launches / one.  Maximum in a sink: 48 x 256 x 512 8.1 / 6.0, 1024 x 256 x 256 8.8 / 6.6, 368 x 384 x 384
// 9.0 / 7.9, 192 x 512 x 512 9.9 / 9.3.  Maximum of its own: 48 x 256 x 512 8.3 / 6.1, 192 x 256 x 256 8.4 / 7.6; a call with its host time
// 12.2 / 7.6 and 12.3 / 7.6.  (Four waves in all, bias and tensor scale loaded behind the product, divisions in the addresses.  In
// a block of 192 rows, dim 256, the output projection took 7.5 us so, now 6.1, FFN down with its 512 columns 10.2, now 8.4.)
#include "ll_common.h"
#include "gemm_epilogue.h"
#include "amax_exchange.h"
#include "norm_rows.h"       // from here on without floating-point contraction
#include "quantize_block.h"

namespace ll {

// Eight waves normalize and quantize; all of them multiply where rows are normalized, four of them otherwise: with more columns per
// workgroup fewer compute units are busy (48 x 256 x 512 7.2 instead of 6.1 us).
constexpr int kFusedThreads = 512;
constexpr int kFusedRows = 32;  // of a workgroup's tile: a wave multiplies all rows and 32 columns
constexpr int kFusedMaxK = 512, kNormMaxK = LL_NORM_GEMM_MAX_C;
constexpr int kFusedPatch = 32 * (64 + 16);       // bytes of a wave's patch in the epilogue

struct FusedParams {
  const uint16_t* x;
  int64_t ldx;
  const unsigned long long* sink_parts;  // null: the maximum of x itself
  uint32_t sink_epoch;
  const uint32_t* sink_epoch_offset;
  const uint8_t *Bv, *Bs;
  const float* amax_b;
  float inv_denom_a, inv_denom_b;
  int M, N, K, Np;
  Divisor tiles_m, row_blocks;  // blocks of 16 of a row
  uint16_t* D;
  int64_t ldd;
  GemmEpilogue epi;
};
// The rows are normalized first: adaLN modulation (a, b: scale and shift, a row per frame) or LayerNorm (weight and bias, or null),
// for up to kMaxGemmGroups products of tiles_n_each column tiles each.
struct NormFusedParams : FusedParams {
  const uint16_t *a, *b;
  int64_t a_stride, b_stride;
  Divisor frame_rows, tiles_n_each;
  int add_one;
  float eps;
  AmaxSink exchange;
  uint32_t spin_limit;
  int recompute;
  GemmGroup more[kMaxGemmGroups - 1];
  // of whole rows of up to kNormMaxK results, see ll_row_norm
  ll_row_norm row_norm[kMaxGemmGroups];
  float row_eps;
  const float *cosp, *sinp;
  int seq_len;
};
enum { kPlainRows, kAdalnRows, kLayerNormRows };
template <int ROWS>
struct FusedParamsOf {
  typedef NormFusedParams type;
};
template <>
struct FusedParamsOf<kPlainRows> {
  typedef FusedParams type;
};
constexpr int fused_cols(int rows) { return rows == kPlainRows ? 128 : 256; }      // of a workgroup: 32 per wave
constexpr int fused_waves(int rows) { return rows == kPlainRows ? 2 : 4; }  // per SIMD: two workgroups with an exchange are resident
constexpr int kExchangeSlots = kAmaxParts / 2;  // of a sink: a launch whose workgroups exchange maxima leaves its results' in the others

// T: 64 elements of K at most, a wave's weights in registers.  Quantization is the arithmetic of quantize_kernel, the product
// the order of gemm_w4a4_kernel<1, 1> (64 elements of K after 64, dword after dword of the lanes' pieces): the same bits.
// Bound by the chain: one trip to memory for x, weights and maximum together, the scale table, a few hundred instructions per
// block of 16 (229 a block and lane), the products, the store.
//
// ROWS other than kPlainRows: the rows are normalized here too, and the tensor maximum is exchanged between the row tiles
// (amax_exchange.h); for the pairs adaLN - q / k / v or FFN up and norm3 - cross-attention q of a small model's block, a launch of 5 to 6 us
// each.  Every column tile normalizes its rows again, 32 rows on one compute unit, so the instructions of a row count: rows
// of up to 256 elements lie two to a wave (norm_rows.h, the same bits), four more waves join in up to the products.  A
// block of 192 rows, dim 256, in two launches each 90.2 us, with a wave per row and four waves 92, with eight 85, so 80.1; of 768
// rows 104.3 / 97.2.  Of 192 rows, dim 512 (a wave per row, eight waves): 108 / 115, hence kNormMaxK.
// Where a workgroup has whole rows of a product, WanRMSNorm and RoPE of q and k follow in the launch (row_norm): that block issues
// two launches less, 8 us of its host time, and takes 79 instead of 82 us, one of 2688 rows 136 instead of 145.  Its 12 us by
// phase: arguments and addresses 1.0, loads 0.9, norm 1.1, exchange 2.1, scale table 0.4, quantization 1.1, product 1.2, rows to LDS
// 1.0, their norm 1.0, and the launch.
template <int RULE, int T, int ROWS>
__global__ __launch_bounds__(kFusedThreads, fused_waves(ROWS)) void quantize_gemm_kernel(typename FusedParamsOf<ROWS>::type p) {
  constexpr bool kNorm = ROWS != kPlainRows;
  constexpr int kRowPitch = 128 * T + 16, kWaveRows = kFusedRows / (kFusedThreads / 64);
  __shared__ __attribute__((aligned(16))) uint8_t s_rows[kNorm ? kFusedRows * kRowPitch : 16];  // normalized, bf16
  __shared__ AmaxExchangeSmem s_exchange;
  constexpr int kPitch = 32 * T + 16, kScalePitch = 4 * T + 2;
  constexpr int kRowBlocks = 4 * T, kBlocks = (kFusedRows * kRowBlocks + kFusedThreads - 1) / kFusedThreads;  // per row; per thread, at most
  __shared__ float s_red[kFusedThreads / 64];
  __shared__ ScaleEntry s_tab[128];
  __shared__ __attribute__((aligned(16))) uint8_t s_values[kFusedRows * kPitch];
  __shared__ __attribute__((aligned(16))) uint8_t s_scales[kFusedRows * kScalePitch];
  __shared__ __attribute__((aligned(16))) uint8_t s_patch[fused_cols(ROWS) / 32 * kFusedPatch];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, lh = lane >> 5;
  GemmGroup pr{p.Bv, p.Bs, nullptr, p.amax_b, p.inv_denom_b, p.D, p.ldd, p.epi.bias, p.epi.sink};
  int tile_n = blockIdx.x / p.tiles_m;
  const int tile_m = blockIdx.x - tile_n * p.tiles_m.d;
  ll_row_norm row_norm{};
  if constexpr (kNorm) {
    const int g = (uint32_t)tile_n / p.tiles_n_each;
    tile_n -= g * p.tiles_n_each.d;
    if (g > 0) pr = p.more[g - 1];
    row_norm = p.row_norm[g];
  }
  const int row0 = tile_m * kFusedRows, col0 = tile_n * fused_cols(ROWS) + 32 * wave;
  const int steps = p.K >> 6;

  // ---- everything the workgroup reads, asked for at once and without branches
  // the thread's blocks of x: block tid + 256 i of the tile's 32 rows
  u32x4 lo[kBlocks], hi[kBlocks];
  int block_row[kBlocks], block_col[kBlocks];
#pragma unroll
  for (int i = 0; i < kBlocks; ++i) {
    const int b = tid + i * kFusedThreads;
    block_row[i] = (uint32_t)b / p.row_blocks;
    block_col[i] = b - block_row[i] * p.row_blocks.d;
    if constexpr (kNorm) continue;
    const int row = min(row0 + block_row[i], p.M - 1);
    const u32x4* src = reinterpret_cast<const u32x4*>(p.x + (int64_t)row * p.ldx + block_col[i] * 16);
    lo[i] = src[0];
    hi[i] = src[1];
  }
  // normalized rows: the wave's four rows of the tile, two pairs (behind the last row: the last again), with their operands
  constexpr int kPairs = kWaveRows / 2;
  uint4 xraw[kPairs][1], araw[kPairs][1], braw[kPairs][1];
  if constexpr (kNorm) {
    const int nchunks = p.K >> 3;
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
      const int row = min(row0 + wave * kWaveRows + 2 * i + lh, p.M - 1);
      load_row<1>(p.x + (int64_t)row * p.ldx, nchunks, l32, xraw[i]);
      if constexpr (ROWS == kAdalnRows) {
        const int f = (uint32_t)row / p.frame_rows;
        load_row<1>(p.a + f * p.a_stride, nchunks, l32, araw[i]);
        load_row<1>(p.b + f * p.b_stride, nchunks, l32, braw[i]);
      }
    }
    if constexpr (ROWS == kLayerNormRows) load_affine<1>(p.a, p.b, nchunks, l32, araw[0], braw[0]);
  }
  // the wave's weights: row l32 of its 32, pieces 2 t + lh of 16 bytes and the scales of their two blocks
  uint4 bv[T];
  uint32_t bs[T];
  if (wave < fused_cols(ROWS) / 32) {
    const int n = min(col0 + l32, p.Np - 1);
    const uint8_t* values = pr.Bv + (int64_t)n * (p.K >> 1) + 16 * lh;
    const uint8_t* scales = pr.Bs + (int64_t)(n >> 7) * (p.K >> 6) * 512 + (n & 31) * 16 + ((n & 127) >> 5) * 4 + 2 * lh;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int at = min(t, steps - 1);
      bv[t] = *reinterpret_cast<const uint4*>(values + 32 * at);
      bs[t] = *reinterpret_cast<const uint16_t*>(scales + 512 * at);
    }
  }
  // and what the epilogue needs
  const float amax_b = pr.amax_b[0];
  EpilogueBias bias_bits;
  if (ROWS == kPlainRows) bias_bits = epilogue_bias<1>(pr.bias, lane, col0, p.N);
  float part = 0.0f, amax;
  if constexpr (kNorm) {
    __builtin_amdgcn_sched_barrier(0);  // all loads are under way
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
      uint4 packed[1];
      if constexpr (ROWS == kAdalnRows)
        part = fmaxf(part, adaln_loaded_row<1, true>(xraw[i], araw[i], braw[i], nullptr, nullptr, p.K, p.eps, p.add_one, l32, packed));
      else
        part = fmaxf(part, layernorm_loaded_row<1, true>(xraw[i], araw[0], braw[0], nullptr, nullptr, p.K, p.eps, l32, packed));
      if (l32 < p.K >> 3) *reinterpret_cast<uint4*>(s_rows + (wave * kWaveRows + 2 * i + lh) * kRowPitch + 16 * l32) = packed[0];
    }
    // The column tiles of a row have the same maximum and share its slot.
    amax = exchange_amax(p.exchange, p.tiles_m.d, (uint32_t)tile_m, part, p.spin_limit, p.recompute != 0, s_exchange, [&](uint32_t s) {
      float m = 0.0f;
#pragma unroll 1
      for (int i = 0; i < kWaveRows; ++i) {
        const int row = min((int)s * kFusedRows + wave * kWaveRows + i, p.M - 1);
        uint4 packed[1];
        if constexpr (ROWS == kAdalnRows) {
          const int f = (uint32_t)row / p.frame_rows;
          m = fmaxf(m, adaln_row<1>(p.x + (int64_t)row * p.ldx, p.a + f * p.a_stride, p.b + f * p.b_stride, p.K, p.eps, p.add_one, lane, packed));
        } else {
          m = fmaxf(m, layernorm_row<1>(p.x + (int64_t)row * p.ldx, p.a, p.b, p.K, p.eps, lane, packed));
        }
      }
      return m;
    });
  } else if (p.sink_parts) {
    const uint32_t epoch = amax_sink_epoch(p.sink_epoch, p.sink_epoch_offset);
#pragma unroll
    for (int i = 0; i < kAmaxParts / kFusedThreads; ++i) part = fmaxf(part, amax_sink_read(p.sink_parts, epoch, i * kFusedThreads + tid));
  } else {
    // eight pieces of 16 bytes under way; behind the end the last one again
    const uint32_t row_pieces = (uint32_t)p.K >> 3, pieces = (uint32_t)p.M * row_pieces;
    for (uint32_t c0 = tid; c0 < pieces; c0 += 8 * kFusedThreads) {
      uint4 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t c = min(c0 + i * kFusedThreads, pieces - 1), r = c / row_pieces;
        v[i] = *reinterpret_cast<const uint4*>(p.x + (int64_t)r * p.ldx + (c - r * row_pieces) * 8);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) part = abs_max_bf16x8(v[i], part);
    }
  }
  if constexpr (!kNorm) {
    part = wave_max(part);
    if (lane == 0) s_red[wave] = part;
    __syncthreads();
    amax = s_red[0];
#pragma unroll
    for (int i = 1; i < kFusedThreads / 64; ++i) amax = fmaxf(amax, s_red[i]);
  }

  // ---- quantization of the 32 rows into LDS (the prologue and the paths of quantize_kernel)
  constexpr bool kStaticRule = (RULE == LL_RULE_STATIC_6 || RULE == LL_RULE_STATIC_4);
  constexpr float kE2 = (RULE == LL_RULE_STATIC_4) ? 4.0f : 6.0f;
  constexpr float kE4 = kStaticRule ? 448.0f : 256.0f;
  const bool fast = amax >= 0x1p-100f && amax <= 0x1p100f;
  const bool approx_ok = amax >= 0x1p-30f && amax <= 0x1p30f;
  const float enc = (kE2 * kE4) / amax;
  const float dec = 1.0f / enc;
  if (fast) fill_scale_table<RULE>(s_tab, amax, dec);
  __syncthreads();
#pragma unroll 1
  for (int i = 0; i < kBlocks; ++i) {
    u32x4 l = lo[0], h = hi[0];
    int row = block_row[0], col = block_col[0];
#pragma unroll
    for (int j = 1; j < kBlocks; ++j)
      if (i == j) l = lo[j], h = hi[j], row = block_row[j], col = block_col[j];
    if (row >= kFusedRows) break;
    if constexpr (kNorm) {
      const u32x4* src = reinterpret_cast<const u32x4*>(s_rows + row * kRowPitch + col * 32);
      l = src[0];
      h = src[1];
    }
    float X[16];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t w = j < 4 ? l[j] : h[j - 4];
      X[2 * j] = __uint_as_float(w << 16);
      X[2 * j + 1] = __uint_as_float(w & 0xFFFF0000u);
    }
    uint32_t out_lo, out_hi, sb;
    if (!fast || !quantize_block_fast<RULE>(X, enc, s_tab, approx_ok, __builtin_inff(), out_lo, out_hi, sb))
      quantize_block<RULE>(X, amax, enc, dec, out_lo, out_hi, sb);
    *reinterpret_cast<uint2*>(s_values + row * kPitch + col * 8) = make_uint2(out_lo, out_hi);
    s_scales[row * kScalePitch + col] = (uint8_t)sb;
  }
  __syncthreads();
  if ((wave >= fused_cols(ROWS) / 32 || col0 >= p.N) && !row_norm.weight) return;

  // what the rows need behind the product, on its way under it
  uint4 row_weight[1];
  uint2 row_bias[4];
  if constexpr (kNorm) {
    if (!row_norm.weight) bias_bits = epilogue_bias<1>(pr.bias, lane, col0, p.N);
  }
  float4 row_cos[kPairs], row_sin[kPairs];
  if constexpr (kNorm) {
    if (row_norm.weight) {
      load_row<1>(static_cast<const uint16_t*>(row_norm.weight), p.N >> 3, l32, row_weight);
#pragma unroll
      for (int rg = 0; rg < 4; ++rg)  // N is a multiple of 8
        row_bias[rg] = *reinterpret_cast<const uint2*>(pr.bias ? pr.bias + min(col0 + 8 * rg + 4 * lh, p.N - 4) : reinterpret_cast<const uint16_t*>(&g_gemm_zero16));
#pragma unroll
      for (int i = 0; i < kPairs; ++i) {
        const int row = row0 + wave * kWaveRows + 2 * i + lh;
        row_cos[i] = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        row_sin[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (row_norm.rope && row < p.seq_len) {
          row_cos[i] = *reinterpret_cast<const float4*>(p.cosp + (int64_t)row * 64 + (l32 & 15) * 4);
          row_sin[i] = *reinterpret_cast<const float4*>(p.sinp + (int64_t)row * 64 + (l32 & 15) * 4);
        }
      }
    }
  }
  // ---- product: 32 x 32 per wave
  float16v acc[1][1];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[0][0][i] = 0.0f;
  const uint8_t* a_values = s_values + l32 * kPitch + 16 * lh;
  const uint8_t* a_scales = s_scales + l32 * kScalePitch + 2 * lh;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    if (t >= steps) break;
    const uint4 av = *reinterpret_cast<const uint4*>(a_values + 32 * t);
    const half2v as = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(*reinterpret_cast<const uint16_t*>(a_scales + 4 * t), 1.0f, false);
    const half2v ws = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(bs[t], 1.0f, false);
    const uint32_t a[4] = {av.x, av.y, av.z, av.w}, b[4] = {bv[t].x, bv[t].y, bv[t].z, bv[t].w};
#pragma unroll
    for (int j = 0; j < 4; ++j)
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode8(b[j], half2v{ws[j >> 1], ws[j >> 1]}),
                                                         decode8(a[j], half2v{as[j >> 1], as[j >> 1]}), acc[0][0], 0, 0, 0);
  }
  const float alpha = (amax * amax_b) * (p.inv_denom_a * pr.inv_denom_b);
  GemmEpilogue epi = p.epi;
  epi.sink = pr.sink;
  uint32_t slot = (uint32_t)blockIdx.x * (kFusedThreads / 64) + wave;
  if (kNorm) slot = kExchangeSlots + slot % (kAmaxParts - kExchangeSlots);
  if constexpr (kNorm) {
    if (row_norm.weight) {
      // The workgroup has whole rows of results: they meet in LDS where the normalized rows were, and every wave takes the rows that
      // it normalized.
      if (col0 < p.N) {
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const int col = col0 + 8 * rg + 4 * lh;
          uint32_t w[2] = {pack_bf16x2(acc[0][0][4 * rg] * alpha, acc[0][0][4 * rg + 1] * alpha),
                           pack_bf16x2(acc[0][0][4 * rg + 2] * alpha, acc[0][0][4 * rg + 3] * alpha)};
          if (pr.bias) {
            const uint2 b = row_bias[rg];
            w[0] = pack_bf16x2(__uint_as_float(w[0] << 16) + __uint_as_float(b.x << 16), __uint_as_float(w[0] & 0xFFFF0000u) + __uint_as_float(b.x & 0xFFFF0000u));
            w[1] = pack_bf16x2(__uint_as_float(w[1] << 16) + __uint_as_float(b.y << 16), __uint_as_float(w[1] & 0xFFFF0000u) + __uint_as_float(b.y & 0xFFFF0000u));
          }
          *reinterpret_cast<uint2*>(s_rows + l32 * kRowPitch + col * 2) = make_uint2(w[0], w[1]);
        }
      }
      __syncthreads();
      const int nchunks = p.N >> 3;
      float out_max = 0.0f;
#pragma unroll
      for (int i = 0; i < kPairs; ++i) {
        const int r = wave * kWaveRows + 2 * i + lh, row = row0 + r;
        const uint4 x[1] = {*reinterpret_cast<const uint4*>(s_rows + r * kRowPitch + min(l32, nchunks - 1) * 16)};
        float v[1][8], o8[8];
        unpack_row<1>(x, nchunks, l32, v);
        const float scale = rms_scale<1, true>(v, nchunks, p.N, p.row_eps);
        norm_rope8(v[0], scale, row_weight[0], row_norm.rope && row < p.seq_len, row_cos[i], row_sin[i], o8);
        const uint4 packed = pack8(o8), smooth = smooth_head8(o8);
        if (row < p.M && l32 < nchunks) {
          *reinterpret_cast<uint4*>(pr.D + (int64_t)row * pr.ldd + 8 * l32) = packed;
          out_max = abs_max_bf16x8(packed, out_max);
          if (row_norm.smooth) *reinterpret_cast<uint4*>(static_cast<uint16_t*>(row_norm.smooth) + (int64_t)row * pr.ldd + 8 * l32) = smooth;
        }
      }
      if (pr.sink.parts) {
        out_max = wave_max(out_max);
        if (lane == 0) amax_sink_update(pr.sink, slot, out_max);
      }
      return;
    }
  }
  gemm_epilogue<1, 1, 4>(acc, alpha, s_patch, wave, lane, row0, col0, p.M, p.N, pr.D, pr.ldd, pr.bias, p.epi.act, epi, slot, bias_bits);
}

template <int RULE, int ROWS>
void launch_rows(const typename FusedParamsOf<ROWS>::type& p, unsigned grid, hipStream_t s) {
  if (ROWS != kPlainRows || p.K <= kNormMaxK)
    hipLaunchKernelGGL((quantize_gemm_kernel<RULE, kNormMaxK / 64, ROWS>), dim3(grid), dim3(kFusedThreads), 0, s, p);
  else if constexpr (ROWS == kPlainRows)
    hipLaunchKernelGGL((quantize_gemm_kernel<RULE, kFusedMaxK / 64, ROWS>), dim3(grid), dim3(kFusedThreads), 0, s, p);
}
template <int ROWS>
void launch_quantize_gemm(const typename FusedParamsOf<ROWS>::type& p, int rule, unsigned grid, hipStream_t s) {
  switch (rule) {
    case LL_RULE_STATIC_6: launch_rows<LL_RULE_STATIC_6, ROWS>(p, grid, s); break;
    case LL_RULE_STATIC_4: launch_rows<LL_RULE_STATIC_4, ROWS>(p, grid, s); break;
    case LL_RULE_MAE: launch_rows<LL_RULE_MAE, ROWS>(p, grid, s); break;
    case LL_RULE_MSE: launch_rows<LL_RULE_MSE, ROWS>(p, grid, s); break;
    default: launch_rows<LL_RULE_ABS_MAX, ROWS>(p, grid, s); break;
  }
}

// Whether two ranges of memory have a byte in common (none of them null and long).
inline bool overlap(const void* a, int64_t bytes_a, const void* b, int64_t bytes_b) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return a && b && x < y + (uintptr_t)bytes_b && y < x + (uintptr_t)bytes_a;
}
inline int64_t matrix_bytes(int64_t rows, int64_t cols, int64_t ld) { return 2 * ((rows - 1) * ld + cols); }

}  // namespace ll

extern "C" int ll_nvfp4_quantize_gemm(const void* x, int64_t M, int64_t K, int64_t ldx, int rule, const ll_amax_sink* x_sink, float denom_a,
                                      const uint8_t* B_values, const uint8_t* B_scales, const float* amax_b, float denom_b, int64_t N,
                                      int64_t Np, void* D, int64_t ldd, const ll_gemm_epilogue* epilogue, void* stream) {
  using namespace ll;
  LL_REQUIRE(x && B_values && B_scales && amax_b && D && epilogue, "ll_nvfp4_quantize_gemm: null pointer");
  LL_REQUIRE(M > 0 && K > 0 && N > 0 && ldx >= K && Np % 128 == 0 && N <= Np && ldd >= N && denom_a > 0.f && denom_b > 0.f,
             "ll_nvfp4_quantize_gemm: bad shape M=%lld N=%lld Np=%lld K=%lld ldx=%lld ldd=%lld", (long long)M, (long long)N, (long long)Np,
             (long long)K, (long long)ldx, (long long)ldd);
  LL_REQUIRE(rule >= 0 && rule <= 4, "ll_nvfp4_quantize_gemm: unknown scale rule %d", rule);
  LL_REQUIRE(!x_sink || (x_sink->parts && sink_is_valid(x_sink)), "ll_nvfp4_quantize_gemm: amax sink needs an 8-byte aligned buffer and a non-zero epoch");
  LL_REQUIRE(((reinterpret_cast<uintptr_t>(B_values) | reinterpret_cast<uintptr_t>(B_scales)) & 15) == 0 &&
                 (reinterpret_cast<uintptr_t>(D) & 1) == 0 && (reinterpret_cast<uintptr_t>(epilogue->bias) & 1) == 0,
             "ll_nvfp4_quantize_gemm: operands must be 16-byte, D and bias 2-byte aligned");
  FusedParams p{};
  if (int rc = make_epilogue(*epilogue, N, p.epi)) return rc;
  // Workgroups that begin late still read x and its maximum when others write results and leave their maxima: two launches do not mind
  // where either lies in the place of the other.
  constexpr int64_t kSinkBytes = (int64_t)kAmaxParts * sizeof(uint64_t);
  if (overlap(D, matrix_bytes(M, N, ldd), x, matrix_bytes(M, K, ldx)) ||
      (x_sink && overlap(x_sink->parts, kSinkBytes, epilogue->amax_sink.parts, kSinkBytes)))
    return LL_ENOSUP;
  // Where the launch is ahead of quantization and product of their own.  A workgroup that reads the whole tensor for its maximum: up
  // to 65536 elements (a call with its host time, two launches / one, us: 64 x 512 x 512 12.4 / 9.9, 128 x 512 x 256 12.4 / 11.3; 192 x 512
  // x 512, beyond the line, 12.6 / 12.5 and on the GPU 9.9 / 12.2).
  if (K % 64 != 0 || K > kFusedMaxK || ldx % 8 != 0 || (reinterpret_cast<uintptr_t>(x) & 15) != 0 || M > (1 << 20) || N > (1 << 20) ||
      (!x_sink && M * K > 65536))
    return LL_ENOSUP;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    set_error("ll_nvfp4_quantize_gemm: hipGetDevice failed");
    return LL_ELAUNCH;
  }
  if (int rc = compute_units_of(dev, cus, "ll_nvfp4_quantize_gemm")) return rc;
  if (!product_takes_plain_64x64_tiles(M, N, K, 1, cus)) return LL_ENOSUP;
  // More than one workgroup per unit of the longer rows, whose quantization is then repeated in turn: 1760 x 512 x 512, 220
  // workgroups, 10.6 / 10.1, 2640 x 512 x 512, 332, 12.0 / 13.1; but 5280 x 256 x 256, 330, 10.3 / 8.7.
  constexpr int cols = fused_cols(kPlainRows);
  const int64_t grid = ((M + kFusedRows - 1) / kFusedRows) * ((N + cols - 1) / cols);
  if (K > 256 && grid > cus) return LL_ENOSUP;
  p.x = static_cast<const uint16_t*>(x);
  p.ldx = ldx;
  if (x_sink) {
    p.sink_parts = reinterpret_cast<const unsigned long long*>(x_sink->parts);
    p.sink_epoch = x_sink->epoch;
    p.sink_epoch_offset = x_sink->epoch_offset;
  }
  p.Bv = B_values;
  p.Bs = B_scales;
  p.amax_b = amax_b;
  p.inv_denom_a = 1.0f / denom_a;
  p.inv_denom_b = 1.0f / denom_b;
  p.M = (int)M;
  p.N = (int)N;
  p.K = (int)K;
  p.Np = (int)Np;
  p.tiles_m = divisor((uint32_t)((M + kFusedRows - 1) / kFusedRows));
  p.row_blocks = divisor((uint32_t)K >> 4);
  p.D = static_cast<uint16_t*>(D);
  p.ldd = ldd;
  launch_quantize_gemm<kPlainRows>(p, rule, (unsigned)grid, static_cast<hipStream_t>(stream));
  LL_CHECK_LAUNCH("quantize_gemm_kernel");
  return LL_OK;
}

extern "C" int ll_nvfp4_norm_gemm(const void* x, int64_t M, int C, const void* scale, const void* shift, int64_t scale_stride,
                                  int64_t shift_stride, int64_t frame_rows, int add_one_to_scale, const void* weight, const void* bias, float eps,
                                  int rule, const ll_amax_sink* exchange, int64_t spin_limit, float denom_a, int64_t N, int64_t Np,
                                  int n_products, const ll_gemm_product* products, int activation, const ll_row_norm* row_norms, float row_eps,
                                  const float* cos, const float* sin, int64_t seq_len, void* stream) {
  using namespace ll;
  const char* what = "ll_nvfp4_norm_gemm";
  LL_REQUIRE(x && products && (scale != nullptr) == (shift != nullptr) && !(scale && (weight || bias)), "%s: null pointer, or both kinds of normalization", what);
  LL_REQUIRE(M > 0 && C > 0 && N > 0 && Np % 128 == 0 && N <= Np && denom_a > 0.f && n_products >= 1 && n_products <= kMaxGemmGroups &&
                 (!scale || (frame_rows > 0 && M % frame_rows == 0)),
             "%s: bad shape M=%lld C=%d N=%lld Np=%lld frame_rows=%lld, %d products", what, (long long)M, C, (long long)N, (long long)Np,
             (long long)frame_rows, n_products);
  LL_REQUIRE(rule >= 0 && rule <= 4, "%s: unknown scale rule %d", what, rule);
  LL_REQUIRE(exchange && exchange->parts && sink_is_valid(exchange), "%s: an amax sink (8-byte aligned buffer, non-zero epoch) is required", what);
  LL_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(scale) | reinterpret_cast<uintptr_t>(shift) |
               reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(bias)) & 15) == 0 && scale_stride % 8 == 0 && shift_stride % 8 == 0,
             "%s: inputs must be 16-byte aligned, strides multiples of 8 elements", what);
  NormFusedParams p{};
  for (int i = 0; i < n_products; ++i) {
    const ll_gemm_product& pr = products[i];
    LL_REQUIRE(pr.B_values && pr.B_scales && pr.amax_b && pr.D && pr.ldd >= N && pr.denom_b > 0.f && !pr.alpha,
               "%s: product %d: null pointer, ldd < N or an alpha", what, i);
    LL_REQUIRE(((reinterpret_cast<uintptr_t>(pr.B_values) | reinterpret_cast<uintptr_t>(pr.B_scales)) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(pr.D) & 1) == 0 && (reinterpret_cast<uintptr_t>(pr.bias) & 1) == 0,
               "%s: product %d: operands must be 16-byte, D and bias 2-byte aligned", what, i);
    ll_gemm_epilogue e{};
    e.bias = pr.bias;
    e.activation = activation;
    e.amax_sink = pr.amax_sink;
    GemmEpilogue epi;
    if (int rc = make_epilogue(e, N, epi)) return rc;
    if (i == 0) {
      p.epi = epi;
      p.Bv = pr.B_values;
      p.Bs = pr.B_scales;
      p.amax_b = pr.amax_b;
      p.inv_denom_b = 1.0f / pr.denom_b;
      p.D = static_cast<uint16_t*>(pr.D);
      p.ldd = pr.ldd;
    } else {
      p.more[i - 1] = GemmGroup{pr.B_values, pr.B_scales, nullptr, pr.amax_b, 1.0f / pr.denom_b, static_cast<uint16_t*>(pr.D), pr.ldd, epi.bias, epi.sink};
    }
  }
  if (row_norms) {
    for (int i = 0; i < n_products; ++i) {
      const ll_row_norm& rn = row_norms[i];
      if (!rn.weight) continue;
      LL_REQUIRE(N % 8 == 0 && products[i].ldd % 8 == 0 && activation == LL_ACT_NONE && (!(rn.rope || rn.smooth) || N % 128 == 0) &&
                     (!rn.rope || (cos && sin && seq_len >= 0)),
                 "%s: product %d: a row norm needs N and ldd of whole 16-byte pieces, no activation, heads of 128 and angles for RoPE", what, i);
      LL_REQUIRE(((reinterpret_cast<uintptr_t>(rn.weight) | reinterpret_cast<uintptr_t>(rn.smooth) | reinterpret_cast<uintptr_t>(products[i].D) |
                   reinterpret_cast<uintptr_t>(cos) | reinterpret_cast<uintptr_t>(sin)) & 15) == 0,
                 "%s: product %d: row norm operands must be 16-byte aligned", what, i);
      // a bias at any element, which the product by itself takes, is loaded here by eights of bytes
      if (N > fused_cols(kAdalnRows) || (reinterpret_cast<uintptr_t>(products[i].bias) & 7) != 0) return LL_ENOSUP;
      p.row_norm[i] = rn;
    }
    p.row_eps = row_eps;
    p.cosp = cos;
    p.sinp = sin;
    p.seq_len = (int)(seq_len < M ? seq_len : M);
  }
  // as in ll_nvfp4_quantize_gemm, and the recomputation of a late workgroup's share reads all of it again; the maxima have slots of their own
  const int64_t frames = scale ? M / frame_rows : 1;
  const struct { const void* at; int64_t bytes; } read[] = {{x, matrix_bytes(M, C, C)}, {scale, matrix_bytes(frames, C, scale_stride)},
      {shift, matrix_bytes(frames, C, shift_stride)}, {weight, matrix_bytes(1, C, C)}, {bias, matrix_bytes(1, C, C)}};
  for (int i = 0; i < n_products; ++i)
    for (const auto& r : read)
      if (overlap(products[i].D, matrix_bytes(M, N, products[i].ldd), r.at, r.bytes) ||
          overlap(p.row_norm[i].smooth, matrix_bytes(M, N, products[i].ldd), r.at, r.bytes))
        return LL_ENOSUP;
  if (C % 64 != 0 || C > kNormMaxK || M > (1 << 20) || N > (1 << 20)) return LL_ENOSUP;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    set_error("%s: hipGetDevice failed", what);
    return LL_ELAUNCH;
  }
  if (int rc = compute_units_of(dev, cus, what)) return rc;
  if (!product_takes_plain_64x64_tiles(M, N, C, n_products, cus)) return LL_ENOSUP;
  const int64_t tiles_m = (M + kFusedRows - 1) / kFusedRows, tiles_n = (N + fused_cols(kAdalnRows) - 1) / fused_cols(kAdalnRows);
  const int64_t grid = tiles_m * tiles_n * n_products;
  // Where the launch is ahead of two: while all its workgroups are resident, two per unit (a block of 2688 rows, dim 256, with one per
  // unit 146.6 us, so 142.5, in two launches each 153; of 1536 rows 110.9, 106.3).
  if (grid > 2 * (int64_t)cus || tiles_m > kExchangeSlots) return LL_ENOSUP;
  p.x = static_cast<const uint16_t*>(x);
  p.ldx = C;
  p.inv_denom_a = 1.0f / denom_a;
  p.M = (int)M;
  p.N = (int)N;
  p.K = C;
  p.Np = (int)Np;
  p.tiles_m = divisor((uint32_t)tiles_m);
  p.tiles_n_each = divisor((uint32_t)tiles_n);
  p.row_blocks = divisor((uint32_t)C >> 4);
  p.a = static_cast<const uint16_t*>(scale ? scale : weight);
  p.b = static_cast<const uint16_t*>(scale ? shift : bias);
  p.a_stride = scale_stride;
  p.b_stride = shift_stride;
  p.frame_rows = divisor(scale ? (uint32_t)frame_rows : 1u);
  p.add_one = add_one_to_scale;
  p.eps = eps;
  p.exchange = make_sink(exchange);
  p.spin_limit = spin_limit < 0 ? 0u : (spin_limit > 0x7FFFFFFF ? 0x7FFFFFFFu : (uint32_t)spin_limit);
  p.recompute = spin_limit < 0 ? 1 : 0;
  if (scale) launch_quantize_gemm<kAdalnRows>(p, rule, (unsigned)grid, static_cast<hipStream_t>(stream));
  else launch_quantize_gemm<kLayerNormRows>(p, rule, (unsigned)grid, static_cast<hipStream_t>(stream));
  LL_CHECK_LAUNCH("quantize_gemm_kernel");
  return LL_OK;
}
