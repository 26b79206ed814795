// Row operations shared by the normalization kernels and by the kernel that normalizes and quantizes in one
// launch: one wave computes one row, a lane holds NCH groups of 8 consecutive elements (group lane + 64 i).
// The order of every floating-point operation is part of the result (the sums are not associative), so every
// kernel that needs a row calls these.
#pragma once
#include "ll_common.h"

#pragma clang fp contract(off)

namespace ll {

__device__ __forceinline__ void unpack8(const uint4& v, float (&f)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(w[i] << 16);
    f[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
  }
}
__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = pack_bf16x2(f[2 * i], f[2 * i + 1]);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// Row kernels: one wave per row (no workgroup barrier; a row's sums are wave reductions), four rows per workgroup.  A lane
// holds NCH groups of 8 elements: NCH = 6 covers C = 3072 exactly, 16 anything up to 8192; groups that a row does not have
// cost their loads and the sum all the same, and their registers waves per SIMD, hence kernels for shorter rows in steps of
// a third or less.  us, with kernels of 1, 3, 6, 10 and 16 groups / with these: LayerNorm 7040 x 1024 7.25 / 6.9, 7040 x
// 2048 12.1 / 11.3, 7040 x 4096 24.0 / 20.7, 7040 x 6144 50.4 / 31.6; adaLN 736 x 2048 4.7 / 4.4, 736 x 6144 10.25 / 9.0;
// RMSNorm 2640 x 6144 14.0 / 11.8.
constexpr int kRowThreads = 256;
constexpr int kRowsPerWg = kRowThreads / 64;
constexpr int kMaxChunks = 16;  // 8 elements each: C <= 64 * 16 * 8 = 8192
constexpr int kMaxRowLength = 64 * kMaxChunks * 8;
#define LL_BY_ROW_LENGTH(C, LAUNCH) \
  if ((C) <= 64 * 1 * 8) {          \
    LAUNCH(1);                      \
  } else if ((C) <= 64 * 2 * 8) {   \
    LAUNCH(2);                      \
  } else if ((C) <= 64 * 3 * 8) {   \
    LAUNCH(3);                      \
  } else if ((C) <= 64 * 4 * 8) {   \
    LAUNCH(4);                      \
  } else if ((C) <= 64 * 6 * 8) {   \
    LAUNCH(6);                      \
  } else if ((C) <= 64 * 8 * 8) {   \
    LAUNCH(8);                      \
  } else if ((C) <= 64 * 10 * 8) {  \
    LAUNCH(10);                     \
  } else if ((C) <= 64 * 12 * 8) {  \
    LAUNCH(12);                     \
  } else if ((C) <= 64 * 14 * 8) {  \
    LAUNCH(14);                     \
  } else {                          \
    LAUNCH(kMaxChunks);             \
  }

// The lane's groups of a row, all requested before the first is waited for; behind the row's end its last group once more.
// (With the load of a group under a branch of its own, and its use there, the compiler waits for every group before it asks
// for the next: a row of 3072 was six trips to memory.  us so / now, with kernels for shorter rows: RMSNorm 880 x 3072 4.8
// / 3.9, LayerNorm 2640 x 3072 8.5 / 7.8, adaLN 736 x 1536 4.0 / 3.6, 4096 x 5120 34.3 / 20.3, q and k 2640 x 3072 17.4 /
// 14.6, 4096 x 5120 42.8 / 33.5, adaLN and quantization 736 x 1536 8.6 / 7.75.)
template <int NCH>
__device__ __forceinline__ void load_row(const uint16_t* __restrict__ row, int nchunks, int lane, uint4 (&raw)[NCH]) {
#pragma unroll
  for (int i = 0; i < NCH; ++i) raw[i] = *reinterpret_cast<const uint4*>(row + min(lane + i * 64, nchunks - 1) * 8);
}
// The operands of a row (weight and bias, scale and shift) are asked for with it where that leaves two waves per SIMD or
// more, and else kLateGroups groups at a time where they are used (us, all ahead in one wave per SIMD / so: adaLN 2640 x
// 7168 32.8 / 22.1, 7040 x 7168 67.5 / 42.0).
template <int NCH>
constexpr bool kOperandsAhead = NCH <= 12;
constexpr int kLateGroups = 4;
template <int NCH>
__device__ __forceinline__ void load_late(const uint16_t* __restrict__ row, int nchunks, int lane, int group, uint4 (&raw)[NCH]) {
  if (kOperandsAhead<NCH> || group % kLateGroups != 0) return;
#pragma unroll
  for (int i = group; i < min(group + kLateGroups, NCH); ++i) raw[i] = *reinterpret_cast<const uint4*>(row + min(lane + i * 64, nchunks - 1) * 8);
}
// As floats, zeros behind the row's end; the lane's sum of them.  No branch and no choice here, into which a load would sink.
template <int NCH>
__device__ __forceinline__ float unpack_row(const uint4 (&raw)[NCH], int nchunks, int lane, float (&v)[NCH][8]) {
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const uint32_t keep = lane + i * 64 < nchunks ? 0xFFFFFFFFu : 0u;
    unpack8(make_uint4(raw[i].x & keep, raw[i].y & keep, raw[i].z & keep, raw[i].w & keep), v[i]);
#pragma unroll
    for (int j = 0; j < 8; ++j) sum += v[i][j];
  }
  return sum;
}
template <bool HALF>
__device__ __forceinline__ float row_sum(float v) {
  return HALF ? half_wave_sum_dpp(v) : wave_sum_dpp(v);
}
// adaLN modulation of one row, utils/adaln_triton.py:36-86: LayerNorm without affine in fp32, rounded to bf16,
// times (1 + scale) rounded, plus shift rounded.  `packed[i]` receives the 8 results of group lane + 64 i; the
// return value is the lane's share of the row's absolute maximum.  Two values share a rounding's conversion: adaln_kernel took
// 9.6 us for 2640 x 3072 so (before load_row), with one each 10.2.
// HALF: a row per half of the wave, lane 0 .. 31 of it, NCH = 1: rows of up to 256 elements, the same bits.
template <int NCH, bool HALF = false>
__device__ __forceinline__ float adaln_loaded_row(const uint4 (&xraw)[NCH], uint4 (&sraw)[NCH], uint4 (&hraw)[NCH],
                                                  const uint16_t* __restrict__ scr, const uint16_t* __restrict__ shr, int C, float eps,
                                                  int add_one, int lane, uint4 (&packed)[NCH]) {
  const int nchunks = C >> 3;
  float v[NCH][8];
  const float sum = unpack_row<NCH>(xraw, nchunks, lane, v);
  const float inv_c = 1.0f / (float)C;
  const float mean = row_sum<HALF>(sum) * inv_c;
  float sq = 0.0f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    if (i * 64 < nchunks) {
      const bool in = lane + i * 64 < nchunks;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] -= mean;
        sq += in ? v[i][j] * v[i][j] : 0.0f;
      }
    }
  }
  const float var = row_sum<HALF>(sq) * inv_c;
  const float rstd = 1.0f / sqrtf(var + eps);
  float out_max = 0.0f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    packed[i] = make_uint4(0u, 0u, 0u, 0u);
    load_late<NCH>(scr, nchunks, lane, i, sraw);
    load_late<NCH>(shr, nchunks, lane, i, hraw);
    if (i * 64 < nchunks) {
      float s8[8], h8[8], y[8];
      unpack8(sraw[i], s8);
      unpack8(hraw[i], h8);
      if (add_one) {
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          s8[j] += 1.0f;
          s8[j + 1] += 1.0f;
          round_to_bf16(s8[j], s8[j + 1]);
        }
      }
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        float x0 = v[i][j] * rstd, x1 = v[i][j + 1] * rstd;
        round_to_bf16(x0, x1);
        x0 *= s8[j];
        x1 *= s8[j + 1];
        round_to_bf16(x0, x1);
        y[j] = x0 + h8[j];
        y[j + 1] = x1 + h8[j + 1];
      }
      if (lane + i * 64 < nchunks) packed[i] = pack8(y);
      out_max = abs_max_bf16x8(packed[i], out_max);
    }
  }
  return out_max;
}

template <int NCH>
__device__ __forceinline__ float adaln_row(const uint16_t* __restrict__ xr, const uint16_t* __restrict__ scr,
                                           const uint16_t* __restrict__ shr, int C, float eps, int add_one, int lane,
                                           uint4 (&packed)[NCH]) {
  const int nchunks = C >> 3;
  uint4 xraw[NCH], sraw[NCH], hraw[NCH];
  load_row<NCH>(xr, nchunks, lane, xraw);
  if (kOperandsAhead<NCH>) {
    load_row<NCH>(scr, nchunks, lane, sraw);
    load_row<NCH>(shr, nchunks, lane, hraw);
  }
  __builtin_amdgcn_sched_barrier(0);  // all loads are under way
  return adaln_loaded_row<NCH>(xraw, sraw, hraw, scr, shr, C, eps, add_one, lane, packed);
}

// LayerNorm with optional weight and bias of one row, wan_5b/modules/model.py:101-111 (nn.LayerNorm on bf16
// tensors: statistics and the affine map in fp32, one rounding to bf16 at the end).
template <int NCH, bool HALF = false>
__device__ __forceinline__ float layernorm_loaded_row(const uint4 (&xraw)[NCH], uint4 (&wraw)[NCH], uint4 (&braw)[NCH],
                                                      const uint16_t* __restrict__ w, const uint16_t* __restrict__ b, int C, float eps,
                                                      int lane, uint4 (&packed)[NCH]) {
  const int nchunks = C >> 3;
  float v[NCH][8];
  const float sum = unpack_row<NCH>(xraw, nchunks, lane, v);
  const float inv_c = 1.0f / (float)C;
  const float mean = row_sum<HALF>(sum) * inv_c;
  float sq = 0.0f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    if (i * 64 < nchunks) {
      const bool in = lane + i * 64 < nchunks;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] -= mean;
        sq += in ? v[i][j] * v[i][j] : 0.0f;
      }
    }
  }
  const float var = row_sum<HALF>(sq) * inv_c;
  const float rstd = 1.0f / sqrtf(var + eps);
  float out_max = 0.0f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    packed[i] = make_uint4(0u, 0u, 0u, 0u);
    if (w) load_late<NCH>(w, nchunks, lane, i, wraw);
    if (b) load_late<NCH>(b, nchunks, lane, i, braw);
    if (i * 64 < nchunks) {
      float w8[8], b8[8], y[8];
      unpack8(wraw[i], w8);
      unpack8(braw[i], b8);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = (v[i][j] * rstd) * w8[j] + b8[j];
      if (lane + i * 64 < nchunks) packed[i] = pack8(y);
      out_max = abs_max_bf16x8(packed[i], out_max);
    }
  }
  return out_max;
}

// The weight and bias of a LayerNorm for the lane's groups: ones and zeros where there is none.
template <int NCH>
__device__ __forceinline__ void load_affine(const uint16_t* __restrict__ w, const uint16_t* __restrict__ b, int nchunks, int lane,
                                            uint4 (&wraw)[NCH], uint4 (&braw)[NCH]) {
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    wraw[i] = make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u);
    braw[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  if (kOperandsAhead<NCH> && w) load_row<NCH>(w, nchunks, lane, wraw);
  if (kOperandsAhead<NCH> && b) load_row<NCH>(b, nchunks, lane, braw);
}
template <int NCH>
__device__ __forceinline__ float layernorm_row(const uint16_t* __restrict__ xr, const uint16_t* __restrict__ w,
                                               const uint16_t* __restrict__ b, int C, float eps, int lane,
                                               uint4 (&packed)[NCH]) {
  const int nchunks = C >> 3;
  uint4 xraw[NCH], wraw[NCH], braw[NCH];
  load_row<NCH>(xr, nchunks, lane, xraw);
  load_affine<NCH>(w, b, nchunks, lane, wraw, braw);
  __builtin_amdgcn_sched_barrier(0);  // all loads are under way
  return layernorm_loaded_row<NCH>(xraw, wraw, braw, w, b, C, eps, lane, packed);
}

// 1 / sqrt(mean of squares + eps) of a row (WanRMSNorm, wan_5b/modules/model.py:82-98).
template <int NCH, bool HALF = false>
__device__ __forceinline__ float rms_scale(const float (&v)[NCH][8], int nchunks, int C, float eps) {
  float sq = 0.0f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    if (i * 64 < nchunks) {
#pragma unroll
      for (int j = 0; j < 8; ++j) sq += v[i][j] * v[i][j];
    }
  }
  const float ms = row_sum<HALF>(sq) / (float)C;
  return 1.0f / sqrtf(ms + eps);
}
// A group of a row normalized with scale r and weights w, then rotated by the group's four angles, each step rounded to bf16.
__device__ __forceinline__ void norm_rope8(const float (&v)[8], float r, const uint4& w, bool rotate, const float4& cs, const float4& sn,
                                           float (&o8)[8]) {
  const float cc[4] = {cs.x, cs.y, cs.z, cs.w}, ss[4] = {sn.x, sn.y, sn.z, sn.w};
  float w8[8], y[8];
  unpack8(w, w8);
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    y[j] = v[j] * r;
    y[j + 1] = v[j + 1] * r;
    round_to_bf16(y[j], y[j + 1]);
    y[j] *= w8[j];
    y[j + 1] *= w8[j + 1];
    round_to_bf16(y[j], y[j + 1]);
  }
  if (rotate) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const float a = y[2 * p], b = y[2 * p + 1];
      o8[2 * p] = a * cc[p] - b * ss[p];
      o8[2 * p + 1] = a * ss[p] + b * cc[p];
      round_to_bf16(o8[2 * p], o8[2 * p + 1]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) o8[j] = y[j];
  }
}
// o8 - its mean over the head, which lies in sixteen neighbouring lanes (utils/quant.py:797-798): mean and difference rounded to bf16.
__device__ __forceinline__ uint4 smooth_head8(const float (&o8)[8]) {
  float part = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) part += o8[j];
  const float mean = round_to_bf16(sum_over_16_lanes(part) * (1.0f / 128.0f));
  float s8[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) s8[j] = o8[j] - mean;
  return pack8(s8);
}

}  // namespace ll
