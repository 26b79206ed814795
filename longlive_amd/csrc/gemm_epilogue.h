// What the W4A4 GEMM kernels share: operand decode and the epilogue of a wave.
#pragma once
#include "ll_common.h"

namespace ll {

// sixteen zero bytes in global memory: what lanes load in place of K elements beyond the end of a row
inline __device__ uint4 g_gemm_zero16;

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

// Decode 8 e2m1 codes (one dword) and scale them by the f16 pair (s, s).
__device__ __forceinline__ half8v decode8(uint32_t w, half2v s2) {
  const half2v p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0) * s2;
  const half2v p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1) * s2;
  const half2v p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2) * s2;
  const half2v p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3) * s2;
  half8v r;
  r[0] = p0[0]; r[1] = p0[1]; r[2] = p1[0]; r[3] = p1[1];
  r[4] = p2[0]; r[5] = p2[1]; r[6] = p3[0]; r[7] = p3[1];
  return r;
}

// 0.5 x (1 + tanh(u)) = x / (1 + exp(-2u)),  u = sqrt(2/pi) (x + 0.044715 x^3)  (nn.GELU(approximate="tanh"))
__device__ __forceinline__ float gelu_tanh_f32(float x) {
  const float u2 = x * (1.5957691216057308f + 0.07135481627260025f * (x * x));  // 2u
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * u2));
}

// What the epilogue does to y = bf16(alpha * acc), in this order (each step optional):
//   y = bf16(y + bias[n]);  y = bf16(act(y));  y = bf16(y * gate[m / gate_rows, n]) (only with residual);
//   y = bf16(residual[m, n] + y);  max |y| goes to the amax sink.
struct GemmEpilogue {
  const uint16_t* bias;
  int act;
  const uint16_t* gate;
  int gate_rows;
  int64_t gate_stride;
  const uint16_t* residual;
  int64_t ldr;
  AmaxSink sink;
};

// Epilogue of one wave: acc[g][f][r] holds output row m = row_base + 32 f + lane % 32 and output column
// n = col_base + 32 g + 8 (r / 4) + 4 (lane / 32) + r % 4.  The wave transposes one 32-row slab at a time through its
// own LDS patch (the stages of the main loop are free by now) and writes rows with coalesced 16-byte stores.  BATCH: rows of
// the residual and the gate under way, as many as are measured to pay: with 4 the hand-scheduled tiles spill 12 to 19
// registers and lose 0.5 to 2.5 us (asm8: 2640 x 3072 x 3072 47 / 50).  The persistent kernel, whose 4 x 4 fragments leave none
// to spare (253 spilled), takes 2: 2640 x 3072 x 3072 89 us, with gate and residual 97.5 (with 4 96 and 110.5; 7040 x 14336 x
// 3072 568 and 676, with 4 607 and 785).
//
// The bias, which epilogue_bias asks for: ahead of the epilogue where the registers are there and something is left to wait for.
struct EpilogueBias {
  uint32_t w[4];  // of the lane's eight columns
};
template <int FB>
__device__ __forceinline__ EpilogueBias epilogue_bias(const uint16_t* __restrict__ bias, int lane, int col_base, int N) {
  const int n_lane = col_base + 8 * (lane % (4 * FB));
  EpilogueBias b;
  if (!bias || ((N & 7) == 0 && (reinterpret_cast<uintptr_t>(bias) & 15) == 0)) {
    const uint4 v = *reinterpret_cast<const uint4*>(bias ? bias + min(n_lane, N - 8) : reinterpret_cast<const uint16_t*>(&g_gemm_zero16));
    b.w[0] = v.x, b.w[1] = v.y, b.w[2] = v.z, b.w[3] = v.w;
  } else {
    uint32_t bits[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) bits[i] = bias[min(n_lane + i, N - 1)];  // behind the last column: not used
#pragma unroll
    for (int i = 0; i < 4; ++i) b.w[i] = bits[2 * i] | bits[2 * i + 1] << 16;
  }
  return b;
}
template <int FA, int FB, int BATCH>
__device__ __forceinline__ void gemm_epilogue(float16v (&acc)[FB][FA], float alpha, uint8_t* smem, int wave, int lane, int row_base,
                                              int col_base, int M, int N, uint16_t* __restrict__ D, int64_t ldd,
                                              const uint16_t* __restrict__ bias, int act, const GemmEpilogue& epi,
                                              uint32_t sink_slot, const EpilogueBias& bias_bits) {
  const int l32 = lane & 31, lh = lane >> 5;
  constexpr int kEpiPitch = 64 * FB + 16;  // bytes per slab row: 32*FB bf16 + pad
  uint8_t* ebuf = smem + wave * (32 * kEpiPitch);
  constexpr int kChunksPerRow = 4 * FB;     // 16-byte chunks (8 columns) per slab row
  const int ch = lane % kChunksPerRow;      // this lane's chunk column, the same in every pass
  const int n_lane = col_base + 8 * ch;
  const bool vec_ok = ((ldd & 7) == 0) && ((reinterpret_cast<uintptr_t>(D) & 15) == 0);
  float out_max = 0.0f;
  // Everything that is read here is asked for in batches and without branches: a load under a condition of its own is waited
  // for before the next is issued.  us, so / now: 48 x 512 x 256 with bias 4.7 / 4.3, with bias, gate and residual 5.3 / 4.7, 368 x 2048 x
  // 2048 with bias 9.1 / 8.7, 880 x 3072 x 3072 with all 25.1 / 24.1, 7040 x 3072 x 3072 with all 132.5 / 129.5.
  float bias_f[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    bias_f[2 * i] = __uint_as_float(bias_bits.w[i] << 16);
    bias_f[2 * i + 1] = __uint_as_float(bias_bits.w[i] & 0xFFFF0000u);
  }
  constexpr int kPasses = (32 * kChunksPerRow) / 64, kBatch = kPasses < BATCH ? kPasses : BATCH;
  constexpr bool kAhead = FA == 1 || BATCH >= 4;  // the first batch of a slab is asked for before its results go to LDS
  uint4 rv[kBatch], gv[kBatch];
  auto load_residual = [&](int f, int it0) __attribute__((always_inline)) {  // N % 8 == 0 where there is one
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int m = min(row_base + 32 * f + ((it0 + j) * 64 + lane) / kChunksPerRow, M - 1), n = min(n_lane, N - 8);
      rv[j] = *reinterpret_cast<const uint4*>(epi.residual + (int64_t)m * epi.ldr + n);
      if (epi.gate) gv[j] = *reinterpret_cast<const uint4*>(epi.gate + (int64_t)(m / epi.gate_rows) * epi.gate_stride + n);
    }
  };
#pragma unroll
  for (int f = 0; f < FA; ++f) {
    if (kAhead && epi.residual) load_residual(f, 0);
#pragma unroll
    for (int g = 0; g < FB; ++g)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        *reinterpret_cast<uint2*>(ebuf + l32 * kEpiPitch + (32 * g + 8 * rg + 4 * lh) * 2) =
            make_uint2(pack_bf16x2(acc[g][f][4 * rg] * alpha, acc[g][f][4 * rg + 1] * alpha),
                       pack_bf16x2(acc[g][f][4 * rg + 2] * alpha, acc[g][f][4 * rg + 3] * alpha));
      }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < kPasses; ++it) {
      if ((it > 0 || !kAhead) && it % kBatch == 0 && epi.residual) load_residual(f, it);
      const int row = (it * 64 + lane) / kChunksPerRow;
      const int m = row_base + 32 * f + row;
      uint4 v = *reinterpret_cast<const uint4*>(ebuf + row * kEpiPitch + ch * 16);
      if (m < M && n_lane < N) {
        uint32_t w[4] = {v.x, v.y, v.z, v.w};
        if (bias) {  // bf16 result + bf16 bias, rounded to bf16 (the separate add of the reference)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            w[i] = pack_bf16x2(__uint_as_float(w[i] << 16) + bias_f[2 * i],
                               __uint_as_float(w[i] & 0xFFFF0000u) + bias_f[2 * i + 1]);
          }
        }
        if (act == LL_ACT_GELU_TANH) {  // GELU (tanh form) of the bf16 value, computed in fp32, rounded to bf16
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            w[i] = pack_bf16x2(gelu_tanh_f32(__uint_as_float(w[i] << 16)),
                               gelu_tanh_f32(__uint_as_float(w[i] & 0xFFFF0000u)));
          }
        }
        if (epi.residual) {  // host side guarantees 16-byte aligned rows and N % 8 == 0 for this path
          const uint4 rr = rv[it % kBatch], gg = gv[it % kBatch];
          const uint32_t r[4] = {rr.x, rr.y, rr.z, rr.w};
          if (epi.gate) {
            const uint32_t g[4] = {gg.x, gg.y, gg.z, gg.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
              w[i] = pack_bf16x2(__uint_as_float(w[i] << 16) * __uint_as_float(g[i] << 16),
                                 __uint_as_float(w[i] & 0xFFFF0000u) * __uint_as_float(g[i] & 0xFFFF0000u));
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
            w[i] = pack_bf16x2(__uint_as_float(r[i] << 16) + __uint_as_float(w[i] << 16),
                               __uint_as_float(r[i] & 0xFFFF0000u) + __uint_as_float(w[i] & 0xFFFF0000u));
        }
        if (epi.sink.parts) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const bool lo_ok = n_lane + 2 * i < N, hi_ok = n_lane + 2 * i + 1 < N;
            if (lo_ok) out_max = fmaxf(out_max, fabsf(__uint_as_float(w[i] << 16)));
            if (hi_ok) out_max = fmaxf(out_max, fabsf(__uint_as_float(w[i] & 0xFFFF0000u)));
          }
        }
        uint16_t* dst = D + (int64_t)m * ldd + n_lane;
        if (vec_ok && n_lane + 8 <= N) {
          *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
          for (int i = 0; i < 8 && n_lane + i < N; ++i) dst[i] = (uint16_t)(w[i >> 1] >> (16 * (i & 1)));
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (epi.sink.parts) {  // one atomic per wave
    if constexpr (FA * FB == 16) {  // by permutes: the moves of wave_max cost that kernel 70 more spilled registers and 6 to 10 %
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) out_max = fmaxf(out_max, __shfl_xor(out_max, o, 64));
    } else {
      out_max = wave_max(out_max);
    }
    if (lane == 0) amax_sink_update(epi.sink, sink_slot, out_max);
  }
}

template <int FA, int FB, int BATCH>
__device__ __forceinline__ void gemm_epilogue(float16v (&acc)[FB][FA], float alpha, uint8_t* smem, int wave, int lane, int row_base,
                                              int col_base, int M, int N, uint16_t* __restrict__ D, int64_t ldd,
                                              const uint16_t* __restrict__ bias, int act, const GemmEpilogue& epi,
                                              uint32_t sink_slot) {
  gemm_epilogue<FA, FB, BATCH>(acc, alpha, smem, wave, lane, row_base, col_base, M, N, D, ldd, bias, act, epi, sink_slot,
                               epilogue_bias<FB>(bias, lane, col_base, N));
}

// The kernel-side epilogue of a caller's ll_gemm_epilogue for a product of N columns.
inline int make_epilogue(const ll_gemm_epilogue& e, int64_t N, GemmEpilogue& epi) {
  LL_REQUIRE(e.activation == LL_ACT_NONE || e.activation == LL_ACT_GELU_TANH, "ll_nvfp4_gemm_tnt: unknown activation %d", e.activation);
  epi = GemmEpilogue{};
  epi.bias = static_cast<const uint16_t*>(e.bias);
  epi.act = e.activation;
  LL_REQUIRE(sink_is_valid(&e.amax_sink), "ll_nvfp4_gemm_tnt_fused: amax sink needs 8-byte alignment and a non-zero epoch");
  epi.sink = make_sink(&e.amax_sink);
  if (e.residual) {
    LL_REQUIRE(N % 8 == 0 && e.ldr % 8 == 0 && e.ldr >= N && (reinterpret_cast<uintptr_t>(e.residual) & 15) == 0,
               "ll_nvfp4_gemm_tnt_fused: residual needs N %% 8 == 0, ldr %% 8 == 0 and 16-byte alignment");
    epi.residual = static_cast<const uint16_t*>(e.residual);
    epi.ldr = e.ldr;
    if (e.gate) {
      LL_REQUIRE(e.gate_rows > 0 && e.gate_rows < (1ll << 31) && e.gate_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(e.gate) & 15) == 0,
                 "ll_nvfp4_gemm_tnt_fused: gate needs gate_rows > 0, gate_stride %% 8 == 0 and 16-byte alignment");
      epi.gate = static_cast<const uint16_t*>(e.gate);
      epi.gate_rows = (int)e.gate_rows;
      epi.gate_stride = e.gate_stride;
    }
  } else {
    LL_REQUIRE(!e.gate, "ll_nvfp4_gemm_tnt_fused: a gate needs a residual");
  }
  return LL_OK;
}
// Whether ll_nvfp4_gemm_tnt(_grouped) computes products of these sizes in 64 x 64 tiles, K in ascending order (gemm_w4a4.hip).
bool product_takes_plain_64x64_tiles(int64_t M, int64_t N, int64_t Kp, int n_products, int cus);

// Several products with the same A operand and the same N and K in one launch (the q / k / v projections of one
// activation): the weight, its scales and tensor scale, the bias, the output and the amax sink of the products
// behind the first one.  The column tiles of all products form one row of tiles_n tiles, tiles_n_each per product.
constexpr int kMaxGemmGroups = 4;
struct GemmGroup {
  const uint8_t* Bv;
  const uint8_t* Bs;
  const float* alpha;
  const float* amax_b;
  float inv_denom_b;
  uint16_t* D;
  int64_t ldd;
  const uint16_t* bias;
  AmaxSink sink;
};
struct GemmGroups {
  int n;             // number of products (1: the plain call, `more` unused)
  int tiles_n_each;  // column tiles per product
  GemmGroup more[kMaxGemmGroups - 1];
};


}  // namespace ll
