// The two ends of the DiT for gfx950: the patch embedding (latents -> tokens, wan_5b/modules/causal_model.py:1052-1053,
// 1535) and the output head's linear layer (tokens -> latents, :925-960, :1840-1857), each a bf16 matrix product whose other
// side is a latent tensor [C, F, H, W] that is read or written in place of its patches: no permuted copy exists.
// fp32 accumulation (v_mfma_f32_32x32x16_bf16), bias added in fp32, one rounding.
#include <type_traits>

#include "ll_common.h"

namespace ll {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

struct PatchGrid {
  int f, h, w;     // token grid
  int pt, ph, pw;  // patch
  int F, H, W;     // latent extent; may exceed grid x patch on the embedding's side (cropped)
};

__device__ __forceinline__ bf16x8 load_bf16x8(const uint16_t* p) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p)); }

// ----------------------------------------------------------------------------- patch embedding
// out[m][n] = sum_k patch(m)[k] weight[n][k] + bias[n], k = ((c pt + dt) ph + dh) pw + dw (the order of the convolution
// weight).  A workgroup takes 32 tokens x 128 outputs, a wave 32 x 32: the tokens' patches are gathered into LDS once
// (32 x K, neighbouring threads take neighbouring tokens of a row), the weight (1.2 MB at full width) comes from L2 straight
// into registers, and the result leaves through LDS in whole rows.  Meant for up to about a thousand tokens, where it is bound
// by its launch and the chain of latencies, of which each loop has few: several elements of a patch per wait, weights and bias
// asked for ahead of the gathering.  us, with an element per wait, integer divisions for its place and a wait per value of the
// bias / now: 192 tokens x 64 -> 256 5.6 / 3.5, 368 x 192 -> 1536 9.2 / 5.7, 1173 x 64 -> 1536 7.4 / 4.7, 2640 x 192 -> 3072 27 / 19 (every workgroup
// gathers its patches anew; a copy of them ahead of a library product takes 20 there).
constexpr int kEmbedTokens = 32, kEmbedOutputs = 128, kEmbedMaxK = 896;  // 32 x (896 + 8) x 2 bytes of LDS
constexpr int kEmbedAhead = 4;   // weight fragments under way
constexpr int kEmbedGather = 4;  // elements or pairs of a patch under way per thread

__global__ __launch_bounds__(256) void patch_embed_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ weight,
                                                          const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, PatchGrid g,
                                                          int M, int N, int K, int pairs) {
  extern __shared__ __attribute__((aligned(16))) uint16_t rows[];  // [32][K + 8], then [32][128 + 8] of the result
  const int pitch = K + 8, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, lh = lane >> 5;
  const int m0 = blockIdx.x * kEmbedTokens, n0 = blockIdx.y * kEmbedOutputs;
  // the first weights and the bias are on their way while the patches are gathered
  const uint16_t* wrow = weight + (int64_t)min(n0 + wave * 32 + l32, N - 1) * K + 8 * lh;
  const int steps = K / 16;
  bf16x8 wf[kEmbedAhead];
#pragma unroll
  for (int j = 0; j < kEmbedAhead; ++j) wf[j] = load_bf16x8(wrow + 16 * min(j, steps - 1));
  uint32_t bias_bits[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) bias_bits[i] = (bias ? bias : weight)[min(n0 + wave * 32 + 8 * (i >> 2) + 4 * lh + (i & 3), N - 1)];
  const uint32_t with_bias = bias ? 0xFFFFu : 0u;  // a mask and not a branch, behind which each load would be waited for
  {
    const int r = tid & 31, m = min(m0 + r, M - 1);
    const int fi = m / (g.h * g.w), hi = m / g.w % g.h, wi = m % g.w;
    const int64_t plane = (int64_t)g.H * g.W;
    const uint16_t* corner = x + (int64_t)fi * g.pt * plane + (int64_t)hi * g.ph * g.W + wi * g.pw;
    // Quotients of numbers below kEmbedMaxK by one multiplication: (k + 1/2) / d is at least 1 / (2 d) from a whole number, more
    // than a thousand times the error of the product.
    const float by_pw = 1.0f / (float)g.pw, by_ph = 1.0f / (float)g.ph, by_pt = 1.0f / (float)g.pt;
    auto gather = [&](auto pair) __attribute__((always_inline)) {
      constexpr int kStep = decltype(pair)::value ? 2 : 1;
      using T = std::conditional_t<decltype(pair)::value, uint32_t, uint16_t>;
      for (int k0 = (tid >> 5) * kStep; k0 < K; k0 += 8 * kStep * kEmbedGather) {
        T v[kEmbedGather];
#pragma unroll
        for (int j = 0; j < kEmbedGather; ++j) {  // behind the last element: the last again
          const int k = min(k0 + 8 * kStep * j, K - kStep);
          const int q = (int)(((float)k + 0.5f) * by_pw), s = (int)(((float)q + 0.5f) * by_ph), c = (int)(((float)s + 0.5f) * by_pt);
          const int dw = k - q * g.pw, dh = q - s * g.ph, dt = s - c * g.pt;
          v[j] = *reinterpret_cast<const T*>(corner + ((int64_t)c * g.F + dt) * plane + dh * g.W + dw);
        }
#pragma unroll
        for (int j = 0; j < kEmbedGather; ++j)
          if (const int k = k0 + 8 * kStep * j; k < K) *reinterpret_cast<T*>(rows + r * pitch + k) = v[j];
      }
    };
    if (pairs) gather(std::true_type{});
    else gather(std::false_type{});
  }
  __syncthreads();
  const uint16_t* arow = rows + l32 * pitch + 8 * lh;
  float16v acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  for (int s = 0; s < steps; s += kEmbedAhead) {  // the next fragments are on their way under the products
    bf16x8 next[kEmbedAhead];
    if (s + kEmbedAhead < steps)
#pragma unroll
      for (int j = 0; j < kEmbedAhead; ++j) next[j] = load_bf16x8(wrow + 16 * min(s + kEmbedAhead + j, steps - 1));
#pragma unroll
    for (int j = 0; j < kEmbedAhead; ++j)
      if (s + j < steps) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j], load_bf16x8(arow + 16 * (s + j)), acc, 0, 0, 0);
    if (s + kEmbedAhead >= steps) break;
#pragma unroll
    for (int j = 0; j < kEmbedAhead; ++j) wf[j] = next[j];
  }
  __syncthreads();
  // lane = token l32, registers 4 j + i = output 8 j + 4 lh + i of the wave's 32
  constexpr int kOutPitch = kEmbedOutputs + 8;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = wave * 32 + 8 * j + 4 * lh;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = acc[4 * j + i] + bf16_bits_to_f32((uint16_t)(bias_bits[4 * j + i] & with_bias));
    *reinterpret_cast<uint2*>(rows + l32 * kOutPitch + n) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (tid >> 4) + 16 * i, n = (tid & 15) * 8;
    if (m0 + r < M && n0 + n < N) *reinterpret_cast<uint4*>(out + (int64_t)(m0 + r) * N + n0 + n) = *reinterpret_cast<const uint4*>(rows + r * kOutPitch + n);
  }
}

// ----------------------------------------------------------------------------- head
// out[c][f pt + p][h ph + q][w pw + r] = sum_k y[m][k] weight[n][k] + bias[n], n = ((p ph + q) pw + r) C + c.  N is small
// (192) and K long (3072): a workgroup takes 32 tokens x 64 outputs and its eight waves an eighth of K each, read straight
// from memory, eight steps under way; the parts meet in LDS and are added in a fixed order.  Bound by the chain of latencies; the
// places of the results and the bias are fetched under the first loads.  us, before that and with loads of steps that do not
// exist waited for / now: 192 tokens x 256 9.1 / 4.9, 368 x 1536 14.5 / 10.6, 2640 x 3072 27.6 / 23.1.
constexpr int kHeadTokens = 32, kHeadOutputs = 64, kHeadWaves = 8, kHeadPitch = kHeadTokens;  // 64 KB of LDS

__global__ __launch_bounds__(kHeadWaves * 64) void patch_head_kernel(const uint16_t* __restrict__ y, const uint16_t* __restrict__ weight,
                                                                     const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, PatchGrid g,
                                                                     int M, int N, int K, int C) {
  __shared__ float parts[kHeadWaves][kHeadOutputs * kHeadPitch];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, lh = lane >> 5;
  const int m0 = blockIdx.x * kHeadTokens, n0 = blockIdx.y * kHeadOutputs;
  // steps of 16 dealt in eight runs
  const int steps = K / 16, first = steps * wave / kHeadWaves, last = steps * (wave + 1) / kHeadWaves;
  const uint16_t* arow = y + (int64_t)min(m0 + l32, M - 1) * K + 8 * lh;
  const uint16_t *w0 = weight + (int64_t)min(n0 + l32, N - 1) * K + 8 * lh, *w1 = weight + (int64_t)min(n0 + 32 + l32, N - 1) * K + 8 * lh;
  float16v acc[2];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.0f;
  struct Fragments {  // of four steps
    bf16x8 a[4], w[2][4];
  } f0, f1;
  auto load = [&](int s, Fragments& f) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = 16 * min(s + j, steps - 1);
      f.a[j] = load_bf16x8(arow + k);
      f.w[0][j] = load_bf16x8(w0 + k);
      f.w[1][j] = load_bf16x8(w1 + k);
    }
  };
  auto multiply = [&](int s, const Fragments& f) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (s + j < last) {
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[0][j], f.a[j], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[1][j], f.a[j], acc[1], 0, 0, 0);
      }
  };
  load(first, f0);
  if (first + 4 < last) load(first + 4, f1);
  // Where the thread's results go, and their bias, while the loads are under way: neighbouring lanes store neighbouring tokens
  // of one output.
  constexpr int kMine = kHeadOutputs / (kHeadWaves * 2);
  int64_t at[kMine];
  uint32_t b[kMine];
  {
    const int m = min(m0 + l32, M - 1), fi = m / (g.h * g.w), hi = m / g.w % g.h, wi = m % g.w;
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
      const int n = min(n0 + (tid >> 5) + i * kHeadWaves * 2, N - 1);
      const int c = n % C, q = n / C, r = q % g.pw, s = q / g.pw, dh = s % g.ph, dt = s / g.ph;
      at[i] = (((int64_t)c * g.F + fi * g.pt + dt) * g.H + hi * g.ph + dh) * g.W + wi * g.pw + r;
      b[i] = (bias ? bias : weight)[n];  // weight has K elements and more for each n
      asm volatile("" : "+v"(at[i]));  // here, and not behind the barrier
    }
  }
  for (int s = first; s < last; s += 8) {  // eight steps under way
    multiply(s, f0);
    if (s + 4 >= last) break;
    if (s + 8 < last) load(s + 8, f0);
    multiply(s + 4, f1);
    if (s + 12 < last) load(s + 12, f1);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) parts[wave][(32 * t + 8 * (r >> 2) + 4 * lh + (r & 3)) * kHeadPitch + l32] = acc[t][r];
  __syncthreads();
  const uint32_t with_bias = bias ? 0xFFFFu : 0u;
  uint32_t result[kMine];
#pragma unroll
  for (int i = 0; i < kMine; ++i) {
    const int j = (tid >> 5) + i * kHeadWaves * 2;
    float v = parts[0][j * kHeadPitch + l32];
#pragma unroll
    for (int w = 1; w < kHeadWaves; ++w) v += parts[w][j * kHeadPitch + l32];
    result[i] = f32_to_bf16_bits(v + bf16_bits_to_f32((uint16_t)(b[i] & with_bias)));
  }
#pragma unroll
  for (int i = 0; i < kMine; ++i) asm volatile("" : "+v"(result[i]));  // all sums ahead of the first branch
#pragma unroll
  for (int i = 0; i < kMine; ++i)
    if (m0 + l32 < M && n0 + (tid >> 5) + i * kHeadWaves * 2 < N) out[at[i]] = (uint16_t)result[i];
}

}  // namespace ll

static int patch_grid(const char* what, int F, int H, int W, int pt, int ph, int pw, ll::PatchGrid* g) {
  LL_REQUIRE(pt > 0 && ph > 0 && pw > 0 && F >= pt && H >= ph && W >= pw, "%s: bad latent %d x %d x %d or patch %d x %d x %d", what, F, H, W, pt, ph, pw);
  *g = ll::PatchGrid{F / pt, H / ph, W / pw, pt, ph, pw, F, H, W};
  LL_REQUIRE((int64_t)g->f * g->h * g->w < (1 << 30), "%s: too many tokens", what);
  return LL_OK;
}

extern "C" int ll_patch_embed(const void* x, int channels, int F, int H, int W, int pt, int ph, int pw, const void* weight, const void* bias,
                              int N, void* out, void* stream) {
  using namespace ll;
  PatchGrid g;
  if (int rc = patch_grid("ll_patch_embed", F, H, W, pt, ph, pw, &g)) return rc;
  LL_REQUIRE(x && weight && out && channels > 0 && N > 0, "ll_patch_embed: null pointer or bad shape");
  const int64_t K = (int64_t)channels * pt * ph * pw;
  LL_REQUIRE(((reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(out)) & 15) == 0 && (reinterpret_cast<uintptr_t>(x) & 1) == 0 &&
                 (reinterpret_cast<uintptr_t>(bias) & 1) == 0,
             "ll_patch_embed: weight and out must be 16-byte aligned");
  if (K % 16 || K > kEmbedMaxK || N % 8 || N > kEmbedOutputs * 65535) {
    set_error("ll_patch_embed: takes patches of a multiple of 16 up to %d elements and a multiple of 8 outputs", kEmbedMaxK);
    return LL_ENOSUP;
  }
  const int M = g.f * g.h * g.w;
  const int pairs = pw % 2 == 0 && W % 2 == 0 && (reinterpret_cast<uintptr_t>(x) & 3) == 0;
  const size_t lds = (size_t)kEmbedTokens * ((K > kEmbedOutputs ? K : kEmbedOutputs) + 8) * 2;
  hipLaunchKernelGGL(patch_embed_kernel, dim3((M + kEmbedTokens - 1) / kEmbedTokens, (N + kEmbedOutputs - 1) / kEmbedOutputs), dim3(256), lds,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(weight),
                     static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(out), g, M, N, (int)K, pairs);
  LL_CHECK_LAUNCH("patch_embed_kernel");
  return LL_OK;
}

extern "C" int ll_patch_head(const void* y, int K, const void* weight, const void* bias, int channels, int F, int H, int W, int pt, int ph, int pw,
                             void* out, void* stream) {
  using namespace ll;
  PatchGrid g;
  if (int rc = patch_grid("ll_patch_head", F, H, W, pt, ph, pw, &g)) return rc;
  LL_REQUIRE(y && weight && out && channels > 0 && K > 0, "ll_patch_head: null pointer or bad shape");
  LL_REQUIRE(F == g.f * pt && H == g.h * ph && W == g.w * pw, "ll_patch_head: the latent has to consist of whole patches");
  LL_REQUIRE(((reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(y)) & 15) == 0 && (reinterpret_cast<uintptr_t>(out) & 1) == 0 &&
                 (reinterpret_cast<uintptr_t>(bias) & 1) == 0,
             "ll_patch_head: y and weight must be 16-byte aligned");
  const int64_t N = (int64_t)channels * pt * ph * pw;
  if (K % 16 || N > kHeadOutputs * 65535) {
    set_error("ll_patch_head: K = %d is not a multiple of 16", K);
    return LL_ENOSUP;
  }
  const int M = g.f * g.h * g.w;
  hipLaunchKernelGGL(patch_head_kernel, dim3((M + kHeadTokens - 1) / kHeadTokens, (unsigned)((N + kHeadOutputs - 1) / kHeadOutputs)),
                     dim3(kHeadWaves * 64), 0, static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(y),
                     static_cast<const uint16_t*>(weight), static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(out), g, M, (int)N, K, channels);
  LL_CHECK_LAUNCH("patch_head_kernel");
  return LL_OK;
}
