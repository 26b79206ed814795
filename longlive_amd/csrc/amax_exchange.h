// The workgroups of one resident launch agree on the maximum of a tensor that they produce together: each
// publishes the maximum of its own share into its own slot of an amax sink under the launch's epoch, and each
// waits - a bounded number of looks - until all slots carry that epoch.  A workgroup whose wait runs out (another
// stream may hold compute units for milliseconds, and a workgroup that has not started cannot publish) computes
// the maxima of the missing workgroups' shares itself, through a function the kernel supplies: the same numbers,
// so every workgroup reaches the end with the same result whatever the others do.
#pragma once
#include "ll_common.h"

namespace ll {

struct AmaxExchangeSmem {
  float red[16];                                    // one partial per wave
  float amax;
  int alone;
  unsigned long long missing[kAmaxParts / 64];      // one bit per slot that did not carry the epoch at the last look
};

// Called once, by every thread of the workgroup (at most 16 whole waves).  `thread_part`: the thread's share of the maximum of
// this workgroup's share; `slot` < G <= kAmaxParts: this workgroup's slot; `share_max(s)`: the calling thread's
// part of the maximum of the share of workgroup s, evaluated by all threads of the workgroup together (uniform
// control flow) when s is missing.  spin_limit + 1 looks at most; `everything`: skip the wait and compute all
// shares (tests of that path).  Returns the tensor maximum.  us a look, by slots: up to 64 0.35, 192 0.48, 256 0.55,
// 512 0.81, 672 0.51, 768 0.59 (words of slots that have all arrived are not looked at again).
template <class ShareMax>
__device__ __forceinline__ float exchange_amax(const AmaxSink& sink, uint32_t G, uint32_t slot, float thread_part,
                                               uint32_t spin_limit, bool everything, AmaxExchangeSmem& sm,
                                               ShareMax&& share_max) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n_waves = (blockDim.x + 63) >> 6;
  const uint32_t epoch = amax_sink_epoch(sink.epoch, sink.epoch_offset);
  // Maximum over the workgroup, in every thread.  A launch uses sm for one exchange, and between the two uses of sm.red here is
  // the barrier behind the looks.
  auto over_waves = [&](float v) {
    v = wave_max(v);
    if (lane == 0) sm.red[wave] = v;
    __syncthreads();
    return max_over_16_lanes(sm.red[min(lane & 15, n_waves - 1)]);
  };
  const float mine = over_waves(thread_part);
  if (threadIdx.x == 0) amax_sink_update(sink, slot, mine);

  // Wave 0 looks at the G slots until all carry this launch's epoch.  Bound by the latency of a trip past the L2, hence eight
  // loads of 64 slots under way at a time and no second look at slots that have all arrived: LayerNorm and quantization of
  // 736 x 1536 (192 slots) 8.4 us, with one load under way 9.7; 2640 x 3072 (672 slots) 16.2 against 18.3.  Every step around the
  // looks is a part of that latency too: with maxima over lanes and waves by LDS permutes and a read per wave the same 736 x
  // 1536 took 8.4 instead of 7.6 us, the one-pass quantization of 48 x 256 4.5 instead of 3.9, of 736 x 1536 5.6 instead of 4.95.
  if (wave == 0) {
    constexpr uint32_t kAtOnce = 8;
    const uint32_t n_words = (G + 63) >> 6;
    bool all_here = false;
    float m = 0.0f;
    uint32_t pending = everything ? 0u : (1u << n_words) - 1u;  // words of 64 slots
    if (everything) {
      for (uint32_t k = 0; k < n_words; ++k) {
        const unsigned long long missing = __builtin_amdgcn_ballot_w64(lane + 64 * k < G);
        if (lane == 0) sm.missing[k] = missing;
      }
    }
#pragma unroll 1
    for (uint32_t look = 0; !everything; ++look) {
#pragma unroll 1
      for (uint32_t k0 = 0; k0 < n_words; k0 += kAtOnce) {
        if (((pending >> k0) & ((1u << kAtOnce) - 1u)) == 0u) continue;
        unsigned long long v[kAtOnce];
#pragma unroll
        for (uint32_t j = 0; j < kAtOnce; ++j) {  // behind the last slot: the last again
          const uint32_t s = lane + 64 * (k0 + j);
          v[j] = __hip_atomic_load(sink.parts + (s < G ? s : G - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (uint32_t j = 0; j < kAtOnce; ++j) {
          const uint32_t k = k0 + j;
          if (k >= n_words) break;
          const bool here = (uint32_t)(v[j] >> 32) == epoch;
          if (here) m = fmaxf(m, __uint_as_float((uint32_t)v[j]));
          const unsigned long long missing = __builtin_amdgcn_ballot_w64(!here && lane + 64 * k < G);
          if (lane == 0) sm.missing[k] = missing;
          if (missing == 0ull) pending &= ~(1u << k);
        }
      }
      if (pending == 0u) {
        all_here = true;
        break;
      }
      if (look >= spin_limit) break;
      __builtin_amdgcn_s_sleep(2);
    }
    m = wave_max(m);
    if (lane == 0) {
      sm.amax = m;
      sm.alone = all_here ? 0 : 1;
    }
  }
  __syncthreads();
  float amax = sm.amax;  // the maximum over the workgroups that have arrived
  if (sm.alone) {        // uniform over the workgroup
    float part = 0.0f;
#pragma unroll 1
    for (uint32_t k = 0; k * 64 < G; ++k) {
      const unsigned long long word = sm.missing[k];
      uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)word), hi = __builtin_amdgcn_readfirstlane((uint32_t)(word >> 32));
#pragma unroll 1
      while ((lo | hi) != 0u) {
        const uint32_t bit = lo != 0u ? (uint32_t)__builtin_ctz(lo) : 32u + (uint32_t)__builtin_ctz(hi);
        if (lo != 0u) lo &= lo - 1u; else hi &= hi - 1u;
        part = fmaxf(part, share_max(64 * k + bit));
      }
    }
    amax = fmaxf(amax, over_waves(part));
  }
  return amax;
}

}  // namespace ll
