// Chunk attention over an NVFP4 KV cache for gfx950, with the dequantization fused into the K/V tile
// load:  out = softmax(q k^T * scale) v  over  [ cached tokens (FP4 slots) | current chunk (bf16) ].
//
// Replaces "dequantize the whole cache to bf16, copy the chunk in, call flash attention"
// (wan_5b/modules/causal_model.py:557-567, 628-671, 781; utils/quant.py:731-768).
//
// A workgroup is 8 waves = two per SIMD, in one of two shapes (template parameter WIDE):
//   * one head x 128 queries: wave w owns 32 queries (w & 3) and every second 64-key tile (w >> 2); the two
//     halves of the key range are merged at the end.  Where tiles are few, several workgroups share the key range of each
//     (plan_narrow_split, attention_split.h);
//   * one head x 256 queries: wave w owns 32 queries and walks both 64-key tiles of an iteration, so a decoded
//     tile serves twice as many MFMAs.  A launch of this shape may hand a workgroup whole tiles, parts of the
//     key range of tiles (combined through device memory), or both: attention_split.h.  Where a head's last
//     group of queries fills at most four of the eight waves, the waves without queries do no matrix work and
//     the division counts such a tile as the lighter load it is.
// A wave needs at most 256 registers (64 for O^T, 32 for S^T, 32 for its Q fragments, the rest for tile
// fragments, raw FP4 data and addressing), which is what lets two waves share a SIMD: while one wave converts
// FP4 data or evaluates exponentials, the other one's MFMAs run.  Per iteration all 512 threads decode 128 keys of K and V
// ((e2m1 x e4m3) x slot scale -> bf16: bit for bit the values the reference's fused cache dequantization and
// ll_kv_dequantize_blocks produce, utils/kernel/kv_dequant_cuda.cu:95-106) into LDS, both
// row-major (one row per key), with the same thread layout and the same byte offsets for K and V.  The MFMAs
// compute S^T = K Q^T and O^T = V^T P^T (v_mfma_f32_32x32x16_bf16), so every lane owns one query column: row max /
// row sum need no cross-lane traffic beyond one swap between the wave halves, and the online-softmax rescale is
// a per-lane scalar.  The V^T operand (a lane needs eight consecutive keys of one head-dim column) comes out of
// the row-major tile through ds_read_b64_tr_b16, the LDS read that transposes 16-bit elements across 16 lanes.
#include "ll_common.h"
#include "attention_split.h"

#include <cfloat>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

namespace ll {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int kHeadDim = 128;
constexpr int kTileKeys = 64;                  // keys per wave tile
constexpr int kIterKeys = 2 * kTileKeys;       // keys decoded per iteration (one tile per key-parity)
constexpr int kWgQueries = 128;
constexpr int kWaveQueries = 32;
constexpr int kKPitch = 272;                   // bytes per key row of K in LDS (256 + 16 pad)
constexpr int kVPitch = 288;                   // bytes per key row of V in LDS (256 + 32 pad: four rows of a transposing read hit 32 different banks)
constexpr int kKTileBytes = kTileKeys * kKPitch;
constexpr int kVTileBytes = kTileKeys * kVPitch;
constexpr int kStageBytes = 2 * kKTileBytes + 2 * kVTileBytes;
constexpr int kMaxSlots = 64;
constexpr int kAttnThreads = 512;

struct AttnParams {
  const uint16_t* q;
  int64_t Lq;
  int H;
  const uint64_t *kv_ptrs, *ks_ptrs, *ka_ptrs, *vv_ptrs, *vs_ptrs, *va_ptrs;
  int64_t n_cached, n_new;
  int bts, n_slots;
  float inv_denom;
  const uint16_t *k_new, *v_new;
  float scale_log2;  // softmax scale * log2(e)
  uint16_t* out;
  AmaxSink sink;  // receives max |out| when sink.parts is not null
  int n_qtiles;     // groups of queries per head
  int full_qtiles;  // tile t < H * full_qtiles is (head t / full_qtiles, group t % full_qtiles); the tiles behind are
                    // the heads' last groups, (head t - H * full_qtiles, group full_qtiles)
  // Division of the launch between its d.G workgroups (attention_split.h).  One workgroup per tile is
  // whole_rounds = 1, extra = 0, units = 0; `partials` / `arrivals` serve the split part.
  Division d;
  uint32_t parts;   // 128-query tiles: workgroups that share a tile's key range; p.d.G = tiles * parts
  float* partials;  // [2 G] (256-query tiles) or [G] records of partial_bytes
  int* arrivals;    // [tiles] counters, zero between launches
};

struct SlotTable {
  const uint8_t* kv[kMaxSlots];
  const uint8_t* ks[kMaxSlots];
  const uint8_t* vv[kMaxSlots];
  const uint8_t* vs[kMaxSlots];
  float kg[kMaxSlots];
  float vg[kMaxSlots];
  int last_arrival;  // whether this workgroup completed the tile it just left a partial result for
};

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) { return pack_bf16x2(a, b); }

// max(v[lane], v[lane ^ 32]) in every lane: one v_permlane32_swap (register file only) instead of a
// permute through LDS, whose result would also wait for every LDS read issued before it.
__device__ __forceinline__ float max_over_wave_halves(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);  // r[0] = lower half twice, r[1] = upper half twice
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// The two e4m3 block scales in the low 16 bits of `word`, as f16 pairs (s, s) ready for a packed multiply.
__device__ __forceinline__ void block_scales_f16(uint32_t word, half2v (&s2)[2]) {
  const half2v sc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(word, 1.0f, false);
  s2[0] = half2v{sc[0], sc[0]};
  s2[1] = half2v{sc[1], sc[1]};
}

// f32(t.lo) * g and f32(t.hi) * g with one instruction each: the mixed-precision fused multiply-add widens
// the selected f16 half on the way in (op_sel_hi marks source 0 as f16, op_sel picks its upper half).  The
// addend is -0, which leaves the product untouched, signed zeros included.
__device__ __forceinline__ float widen_mul_lo(half2v t, float g) {
  float r;
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(t), "v"(g), "s"(-0.0f));
  return r;
}
__device__ __forceinline__ float widen_mul_hi(half2v t, float g) {
  float r;
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(t), "v"(g), "s"(-0.0f));
  return r;
}

// 8 e2m1 codes (one dword) of a block with scale s2 = (s, s) and slot scale gs -> the 8 fp32 values
// (code * s) * gs, the expression of the reference's fused cache dequantization (utils/kernel/kv_dequant_cuda.cu:
// 97-106).  code * s has at most six significant bits and lies within [2^-10, 2688], so the packed f16 product is
// exact; the multiplication by gs is the only rounding, done in fp32.
__device__ __forceinline__ void fp4x8_to_f32(uint32_t w, half2v s2, float gs, float (&o)[8]) {
  const half2v t0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0) * s2;
  const half2v t1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1) * s2;
  const half2v t2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2) * s2;
  const half2v t3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3) * s2;
  o[0] = widen_mul_lo(t0, gs); o[1] = widen_mul_hi(t0, gs);
  o[2] = widen_mul_lo(t1, gs); o[3] = widen_mul_hi(t1, gs);
  o[4] = widen_mul_lo(t2, gs); o[5] = widen_mul_hi(t2, gs);
  o[6] = widen_mul_lo(t3, gs); o[7] = widen_mul_hi(t3, gs);
}

// Raw FP4 data prefetched one iteration ahead.  Only packed bytes and scale bytes are held in registers
// across the MFMA phase; everything else (slot scale, kind of key, bf16 source rows of the current chunk)
// is re-derived from the key index when the data is decoded.
struct KRaw {         // K or V of one key, one quarter of the head dimension (32 elements)
  uint4 v;            // 16 packed bytes
  uint16_t scales;    // 2 e4m3 block scales (low 16 bits)
};

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 load_global_b128(const void* ptr) {
  const u32x4 v = load_global<u32x4>(ptr);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// Raw FP4 loads.  vo / so are byte offsets of the thread's data inside the slot's value / scale arrays;
// the caller keeps them up to date incrementally (both advance by a constant per iteration inside a slot).
__device__ __forceinline__ void fetch_row(const uint8_t* values, const uint8_t* scales, uint32_t vo, uint32_t so, KRaw& f) {
  f.v = load_global_b128(values + vo);
  f.scales = load_global<uint16_t>(scales + so);
}

// 16 bytes per lane from global memory (base + offset; the base wave-uniform) straight into LDS at lds_base + 16 * lane.
// An asm statement on purpose: for the builtin the compiler's wait-count pass, which cannot tell the two LDS stages apart,
// makes later LDS reads of the *other* stage wait for the load.  The kernel waits for these loads itself
// (vmcnt(0) ahead of the barrier that hands the stage over).
__device__ __forceinline__ void load_to_lds_b128(uint32_t offset, const void* base, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds_base) : "memory");
}
__device__ __forceinline__ const void* wave_uniform(const void* p) {
  const uint64_t v = (uint64_t)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<const void*>((uintptr_t)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}

// Decode 32 elements of one key (K or V) to bf16 and store the 64 bytes into the key's LDS row.
// kind: 0 = fp4 slot data in f (gs = slot amax * f32(1 / (e2m1_max * e4m3_max))), 1 = bf16 row at src, 2 = zeros.
__device__ __forceinline__ void store_row(const KRaw& f, int kind, float gs, const uint4* src, uint8_t* dst) {
  uint4* d4 = reinterpret_cast<uint4*>(dst);
  if (kind == 0) {
    const uint32_t w[4] = {f.v.x, f.v.y, f.v.z, f.v.w};
    half2v s2[2];
    block_scales_f16(f.scales, s2);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v8[8];
      fp4x8_to_f32(w[j], s2[j >> 1], gs, v8);
      d4[j] = make_uint4(pack_bf16(v8[0], v8[1]), pack_bf16(v8[2], v8[3]), pack_bf16(v8[4], v8[5]), pack_bf16(v8[6], v8[7]));
    }
  } else if (kind == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) d4[i] = src[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) d4[i] = make_uint4(0, 0, 0, 0);
  }
}

// The kernel's arguments, read again from the argument segment at the point of use.  What is needed only between
// two segments of work (output pointers, the split of the units) then occupies no scalar registers during the main
// loops, which need all of them; the empty asm statement keeps the compiler from moving the reads to the kernel's start.
__device__ __forceinline__ const __attribute__((address_space(4))) AttnParams& reread_params() {
  const __attribute__((address_space(4))) AttnParams* a =
      (const __attribute__((address_space(4))) AttnParams*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return *a;
}
// The launch's division as an ordinary value (seven scalar loads from the argument segment).
__device__ __forceinline__ Division division_of(const __attribute__((address_space(4))) AttnParams& c) {
  return Division{c.d.G, c.d.whole_rounds, c.d.extra, c.d.n_iter, c.d.units, c.d.full_units, c.d.light};
}
// threadIdx.x as a value the compiler knows nothing about: what is derived from it inside a segment's prologue or
// epilogue is then computed there, and not ahead of the loop over segments, where it would occupy registers
// throughout the main loops.
__device__ __forceinline__ int fresh_thread_index() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}
// Partial results travel between workgroups on different XCDs, whose L2 caches do not see each other's lines.
// Device-scope relaxed atomic accesses go past the L2 (the stores write through, the loads fetch from memory), so
// the exchange needs no device-scope fence - a fence would write back and invalidate the XCD's whole L2, which at
// that moment holds the K/V tiles the other 31 workgroups of the XCD are working through.
__device__ __forceinline__ void store_shared_f32(float* ptr, float v) {
  __hip_atomic_store(reinterpret_cast<uint32_t*>(ptr), __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_shared_f32(const float* ptr) {
  return __uint_as_float(__hip_atomic_load(reinterpret_cast<const uint32_t*>(ptr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
// The same, sixteen or eight bytes per lane (buffer accesses with the sc1 bit: device scope).
typedef float float4v __attribute__((ext_vector_type(4)));
constexpr int kDeviceScope = 1 << 4;
__device__ __forceinline__ void store_shared_b128(__amdgpu_buffer_rsrc_t mem, uint32_t offset, uint32_t base, float4v x) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), mem, offset, base, kDeviceScope);
}
__device__ __forceinline__ void store_shared_b64(__amdgpu_buffer_rsrc_t mem, uint32_t offset, uint32_t base, float2v x) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), mem, offset, base, kDeviceScope);
}
__device__ __forceinline__ float4v load_shared_b128(__amdgpu_buffer_rsrc_t mem, uint32_t offset, uint32_t base) {
  return __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(mem, offset, base, kDeviceScope));
}
__device__ __forceinline__ float2v load_shared_b64(__amdgpu_buffer_rsrc_t mem, uint32_t offset, uint32_t base) {
  return __builtin_bit_cast(float2v, __builtin_amdgcn_raw_buffer_load_b64(mem, offset, base, kDeviceScope));
}
// This workgroup's number in the order in which the work is handed out: consecutive hardware workgroup numbers go
// to different XCDs; every XCD gets a contiguous range of the work instead, so that workgroups that share an L2
// read the same heads.
__device__ __forceinline__ uint32_t group_number(uint32_t G) {
  uint32_t b = blockIdx.x;
  asm volatile("" : "+s"(b));
  return G % 8 == 0 ? (b & 7) * (G / 8) + (b >> 3) : b;
}

// The wave's results O^T * inv_l (register r of o[d]: column 32 d + 8 (r / 4) + 4 lh + r % 4 of query l32), as bf16, to the
// first `queries` of its 32 rows of 32 N columns at dst (rows H heads apart), through an LDS patch of the wave's own: whole
// rows per store.  Straight from the registers a store reaches 16 bytes of each of 32 rows: 7040 queries x 24 heads over
// 512 keys 71.5 us, so 63.1; 3520 x 24 46.7 / 41.2; 1760 x 12 16.3 / 15.1.  out_max: raised to the largest magnitude.
template <int N>
__device__ __forceinline__ void write_rows(const float16v (&o)[N], float inv_l, uint8_t* patch, int lane, uint16_t* dst, int H, int queries,
                                           float& out_max) {
  constexpr int kPitch = 64 * N + 16, kLanes = 4 * N, kRows = 64 / kLanes;  // lanes per row of 16 bytes each, rows per store
  const int l32 = lane & 31, lh = lane >> 5;
#pragma unroll
  for (int d = 0; d < N; ++d)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)
      *reinterpret_cast<uint2*>(patch + l32 * kPitch + (32 * d + 8 * rg + 4 * lh) * 2) =
          make_uint2(pack_bf16(o[d][4 * rg] * inv_l, o[d][4 * rg + 1] * inv_l), pack_bf16(o[d][4 * rg + 2] * inv_l, o[d][4 * rg + 3] * inv_l));
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int at = (lane % kLanes) * 16;
#pragma unroll
  for (int it = 0; it < 32 / kRows; ++it) {
    const int row = it * kRows + lane / kLanes;
    const uint4 v = *reinterpret_cast<const uint4*>(patch + row * kPitch + at);
    if (row < queries) {
      *reinterpret_cast<uint4*>(reinterpret_cast<uint8_t*>(dst + (int64_t)row * H * kHeadDim) + at) = v;
      out_max = abs_max_bf16x8(v, out_max);
    }
  }
}

// f(0), f(1), ... with every index a constant of its own type.
template <typename F, int... I>
__device__ __forceinline__ void each_index(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

template <bool WIDE>
__global__ __launch_bounds__(kAttnThreads) void kv_attention_kernel(AttnParams p) {
  constexpr int kQueries = WIDE ? 2 * kWgQueries : kWgQueries;  // queries per workgroup
  constexpr int kHalves = WIDE ? 2 : 1;                          // 64-key tiles a wave works through per iteration
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  SlotTable& tab = *reinterpret_cast<SlotTable*>(smem + 2 * kStageBytes);

  const int n_iter = (int)((p.n_cached + p.n_new + kIterKeys - 1) / kIterKeys);
  // 256-query tiles: where this workgroup is in its work (attention_split.h).  With 128 queries it has one segment: its part
  // of the key range of one tile.
  WorkCursor at{};
  if constexpr (WIDE) {
    const auto& c = reread_params();
    at = start_of_work(group_number(c.d.G), division_of(c));
  }

  if (const int tid = threadIdx.x; tid < p.n_slots) {
    tab.kv[tid] = reinterpret_cast<const uint8_t*>(p.kv_ptrs[tid]);
    tab.ks[tid] = reinterpret_cast<const uint8_t*>(p.ks_ptrs[tid]);
    tab.vv[tid] = reinterpret_cast<const uint8_t*>(p.vv_ptrs[tid]);
    tab.vs[tid] = reinterpret_cast<const uint8_t*>(p.vs_ptrs[tid]);
    tab.kg[tid] = load_global<float>(reinterpret_cast<const void*>(p.ka_ptrs[tid])) * p.inv_denom;
    tab.vg[tid] = load_global<float>(reinterpret_cast<const void*>(p.va_ptrs[tid])) * p.inv_denom;
  }

  __syncthreads();

  // After its whole tiles (workgroups that share an XCD run neighbouring tiles of a round side by side, in step
  // through the key range), a workgroup's share of the units is cut at tile boundaries into segments: iterations
  // [seg_begin, seg_end) of one tile (head x group of queries).  A segment that is a whole tile ends with the normalised output; the
  // others leave (O, reference point, row sum) in `partials`, and the workgroup that finishes a tile's last
  // segment combines them.  The segments are taken from the share's end backwards: a share is typically the
  // tail of one tile followed by the head of the next, and with the head (keys from 0) first and the tail
  // (keys up to the end) last, all workgroups of the launch move through the key range together, a few
  // iterations apart at most, which is what lets those of one head find each other's K/V lines in the L2.
  for (;;) {
  int tile_id, seg_begin, seg_end;
  bf16x8 qf[8];
  if constexpr (WIDE) {
    const auto& c = reread_params();
    Segment seg;
    if (!next_segment(at, group_number(c.d.G), division_of(c), seg)) break;
    tile_id = (int)seg.tile;
    seg_begin = seg.begin;
    seg_end = seg.end;
  } else {
    const uint32_t g = group_number(p.d.G), part = g % p.parts;
    tile_id = (int)(g / p.parts);
    seg_begin = first_iteration_of_part(part, p.parts, n_iter);
    seg_end = first_iteration_of_part(part + 1, p.parts, n_iter);
  }
  int head, qtile;
  if (const int n_full = p.H * p.full_qtiles; tile_id < n_full) {
    head = tile_id / p.full_qtiles;
    qtile = tile_id - head * p.full_qtiles;
  } else {
    head = tile_id - n_full;
    qtile = p.full_qtiles;
  }
  // The thread's coordinates, derived anew in every segment (see fresh_thread_index).
  const int tid = fresh_thread_index(), lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, lh = lane >> 5;
  const int qq = WIDE ? wave : (wave & 3), kp = WIDE ? 0 : (wave >> 2);  // group of 32 queries, key parity
  // 256-query kernel: when the tile holds at most 128 queries (the last group of queries of a head is rarely
  // full), its waves 4..7 have none, and each wave that has some then has its SIMD to itself (waves w and w + 4
  // share one).  The waves without queries take their part in bringing K and V into LDS and in every barrier, and
  // nothing else: no MFMAs, no exponentials, no fragment reads.  With more than 128 queries some SIMD carries two
  // busy waves whatever the others do, and nothing would be gained (in the 128-query kernel, where the two waves
  // of a SIMD serve the same queries, never).
  bool wave_idle = false;
  if constexpr (WIDE) {
    const auto& c = reread_params();
    const int64_t first = (int64_t)qtile * kQueries;
    wave_idle = __builtin_amdgcn_readfirstlane((int)(c.Lq - first <= 128 && first + qq * kWaveQueries >= c.Lq)) != 0;
  }
  if constexpr (WIDE) {
    const auto& c = reread_params();
    int64_t query = (int64_t)qtile * kQueries + qq * kWaveQueries + l32;
    if (query >= c.Lq) query = c.Lq - 1;
    const uint16_t* src = c.q + (query * p.H + head) * kHeadDim + 8 * lh;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(src + 16 * ks));
  } else {
    // Four whole rows per load, into a patch of the stage that the first iteration leaves alone; the fragments are read
    // from there behind the loads of the first tile.  Straight into the fragments a load reaches 32 bytes of each of 32
    // rows: 1760 queries x 12 heads over 512 keys 15.1 us, so 13.9.  (256-query tiles: 2640 x 24 over 512 27.8 and 28.4,
    // 3520 x 24 41.1 and 40.5.)
    const auto& c = reread_params();
    const int64_t first_query = (int64_t)qtile * kQueries + qq * kWaveQueries;
    uint8_t* patch = smem + ((seg_begin & 1) ^ 1) * kStageBytes + wave * kWaveQueries * kKPitch;
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int row = it * 4 + (lane >> 4);
      const uint4 v = *reinterpret_cast<const uint4*>(c.q + (min(first_query + row, c.Lq - 1) * p.H + head) * kHeadDim + (lane & 15) * 8);
      *reinterpret_cast<uint4*>(patch + row * kKPitch + (lane & 15) * 16) = v;
    }
  }

  float16v o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
  // The reference point starts below every finite score and not at -inf: a tile whose scores are all -inf leaves it there and
  // weighs exp2(-inf) = 0, where -inf - -inf is NaN.
  float m_run = -FLT_MAX, l_run = 0.0f;

  // ---- decode plan.  Thread = (key_local = tid / 4, quarter of the head dim = tid % 4), the same for K and V.
  // Schedule of iteration `it`: the MFMAs work on LDS stage it & 1 while the raw FP4 bytes of iteration
  // it + 1 (already in registers) are decoded into the other stage during the S phase.  As soon as the raw
  // registers are free the bytes of iteration it + 2 are requested, which gives each load most of an
  // iteration to land.  Position of the data the raw registers hold (or will hold next): iter_base = first
  // key of that iteration; per thread the key iter_base + k_local as (slot, offset in slot) plus the byte
  // offsets of its packed values and scales in the slot, which K and V share.
  KRaw kf, vf;
  const int n_cached = (int)p.n_cached, Lk_i = (int)(p.n_cached + p.n_new);
  const int k_local = tid >> 2, k_quarter = tid & 3;
  const uint32_t row_bytes = (uint32_t)p.H * 64u;
  const uint32_t step_vo = (uint32_t)kIterKeys * row_bytes;
  const uint32_t step_so = (uint32_t)p.H * 1024u;
  const int k_dst_off = (k_local >> 6) * kKTileBytes + (k_local & 63) * kKPitch + k_quarter * 64;
  const int v_dst_off = 2 * kKTileBytes + (k_local >> 6) * kVTileBytes + (k_local & 63) * kVPitch + k_quarter * 64;
  int iter_base = seg_begin * kIterKeys;
  int k_slot = (iter_base + k_local) / p.bts, k_off = iter_base + k_local - k_slot * p.bts;
  uint32_t k_vo, k_so;
  float k_gs, v_gs;  // slot scale amax * f32(1 / (e2m1_max * e4m3_max)) of the thread's key, for K and for V
  auto locate = [&]() __attribute__((always_inline)) {
    const int64_t row = (int64_t)k_off * p.H + head;
    k_vo = (uint32_t)row * 64u + k_quarter * 16u;
    k_so = (uint32_t)blocked_scale_offset(row, k_quarter * 2, 8);
    k_gs = tab.kg[min(k_slot, kMaxSlots - 1)];
    v_gs = tab.vg[min(k_slot, kMaxSlots - 1)];
  };
  locate();
  auto fetch_next = [&]() __attribute__((always_inline)) {
    if (iter_base + k_local < n_cached) {
      fetch_row(tab.kv[k_slot], tab.ks[k_slot], k_vo, k_so, kf);
      fetch_row(tab.vv[k_slot], tab.vs[k_slot], k_vo, k_so, vf);
    }
  };
  auto advance = [&]() __attribute__((always_inline)) {
    iter_base += kIterKeys;
    k_off += kIterKeys;
    k_vo += step_vo;
    k_so += step_so;
    if (k_off >= p.bts) {
      do {
        k_off -= p.bts;
        ++k_slot;
      } while (k_off >= p.bts);
      locate();
    }
  };
  auto decode_any = [&](int stage) __attribute__((always_inline)) {
    const int key = iter_base + k_local;
    const int kind = key < n_cached ? 0 : (key < Lk_i ? 1 : 2);
    const int64_t src_off = ((int64_t)(key - n_cached) * p.H + head) * kHeadDim + k_quarter * 32;
    store_row(kf, kind, k_gs, reinterpret_cast<const uint4*>(p.k_new + src_off), smem + stage * kStageBytes + k_dst_off);
    store_row(vf, kind, v_gs, reinterpret_cast<const uint4*>(p.v_new + src_off), smem + stage * kStageBytes + v_dst_off);
  };

  // Reference point of the exponentials.  m_run is not the exact running maximum: it is raised only when
  // the maximum has grown by more than kRescaleStep (in the exp2 domain) since it was last raised, so P can
  // reach 2^kRescaleStep instead of 1 (harmless in fp32 / bf16) and the 64 accumulator registers per lane
  // are rescaled a handful of times per kernel instead of at almost every tile.  The final division by
  // the row sum, which is accumulated against the same reference, makes the result independent of it.
  // Where workgroups share the key range of a 128-query tile the step is 2^2, as for the short launches: the result is then no
  // further from fp64 than that of the 256-query tiles' shares, which it replaced (736 queries x 12 heads over 2208 keys 0.002287
  // relative, 2-norm, against 0.002302; with 2^8 0.002318).
  const float kRescaleStep = !WIDE && p.parts > 1 ? 2.0f : 8.0f;

  // Second half of an iteration: reference point of the exponentials over the wave's 64 keys (S^T in sc:
  // register r of tile kt <-> key 32 kt + 8 (r / 4) + 4 lh + r % 4), then the PV phase in four steps of 16
  // keys, the exponentials of step j + 1 computed under the four MFMAs of step j.
  auto softmax_pv = [&](float16v (&sc)[2], const uint8_t* vt_base) __attribute__((always_inline)) {
    // V^T fragment of step `step` (16 keys), head-dim tile dt: lane l needs column d = 32 dt + l % 32 for the keys
    // 16 step + 8 j + 4 (l / 32) + 0..3 (j = 0, 1: the order of P's registers).  One transposing read serves a
    // 16-lane group: source lane i points at row key0 + i / 4, columns d0 + 4 (i % 4) .. + 3, and every lane of
    // the group receives column d0 + i of the four rows.
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) bf16x4* lds_bf16x4_t;
    const uint8_t* vt_lane = vt_base + (4 * lh + ((lane & 15) >> 2)) * kVPitch + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
    auto read_v = [&](int step, bf16x4 (&dst)[4][2]) __attribute__((always_inline)) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          dst[dt][j] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (lds_bf16x4_t)(vt_lane + (16 * step + 8 * j) * kVPitch + dt * 64));
    };
    bf16x4 vfr[2][4][2];
    read_v(0, vfr[0]);
    __builtin_amdgcn_sched_barrier(0);
    float neg;
    {
      float mx = sc[0][0];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[kt][r]);
      mx = max_over_wave_halves(mx);
      const bool raise = (mx - m_run) * p.scale_log2 > kRescaleStep;
      const float m_new = raise ? mx : m_run;
      const float alpha = raise ? __builtin_amdgcn_exp2f((m_run - m_new) * p.scale_log2) : 1.0f;
      neg = -m_new * p.scale_log2;
      m_run = m_new;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
      }
    }
    float sum = 0.0f;
    auto make_p = [&](int step, bf16x8& dst) __attribute__((always_inline)) {
      const int kt = step >> 1, hf = step & 1;
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[kt][8 * hf + 2 * i], p.scale_log2, neg));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[kt][8 * hf + 2 * i + 1], p.scale_log2, neg));
        sum += p0 + p1;
        w[i] = pack_bf16(p0, p1);
      }
      dst = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
    };
    // The scheduling barriers keep every LDS read where it is written: a whole step ahead of the MFMAs that use
    // it.  Left alone, the compiler moves each read down to just ahead of its MFMA to shorten register live
    // ranges, and the wave then sits out the LDS latency a dozen times per tile.
    bf16x8 pb[2];
    make_p(0, pb[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int step = 0; step < 4; ++step) {
      if (step < 3) read_v(step + 1, vfr[(step + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const bf16x4(&v)[2] = vfr[step & 1][dt];
        const bf16x8 a = __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pb[step & 1], o[dt], 0, 0, 0);
      }
      if (step < 3) {
        make_p(step + 1, pb[(step + 1) & 1]);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
          __builtin_amdgcn_sched_group_barrier(0x400, 2, 0);  // two exponentials
          __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);  // their multiply-adds, sums and packing
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l_run += sum;
  };

  // 256-query tiles, iterations whose 128 keys are all there: 64 slots of one MFMA with what is to run beside it, held in place by
  // scheduling barriers, in which no instruction waits for another.  S^T of both tiles of 64 keys comes first, then O^T of both;
  // the probabilities of the first tile are formed under the second S^T, those of the second under the first O^T, and the next
  // iteration's K and V are converted under the first S^T and the second O^T.
  // The reference point is softmax_pv's, bit for bit, without a maximum per tile: while the probabilities that a lane has of a tile
  // add up to no more than 128, none of them is above 2^7, and softmax_pv would have raised nothing.  Where they add up to more (a
  // segment's first tile and a handful behind it; NaN, too) follow_maximum does what softmax_pv does and forms the tile's
  // probabilities again, and it is to be reached before the first of them is multiplied: hence this order.
  // What bounds the loop is the power limit: the MFMA pipe is busy 59 % of the cycles at 1.74 GHz with 7.1 vector instructions per
  // MFMA, where with a maximum per tile it was 54 % at 1.81 GHz with 8.0, so what counts is what is not executed.  Raw bytes are
  // asked for without branches, behind which the compiler waits for every load under way.  us, with a maximum per tile and the
  // softmax in a burst behind each S^T / so: 2640 queries x 24 heads over 10560 cached + 2640 keys 419 / 404, 7040 x 24 over 21120 +
  // 7040 2254 / 2152, 2328 x 16 over 9312 + 2328 232 / 221; where a key far above the others raises the reference point every
  // fourth iteration, the first shape 398 / 392.  With the packing left to the compiler, which sinks it behind the branch, so
  // that 32 values stay in place of 16, 453.  The kernel then takes all 256 registers; the thread's index waits in scratch memory
  // for the segment's end.
  int it = seg_begin;
  auto wide_iteration = [&](auto convert_tag) __attribute__((always_inline)) {
    constexpr bool kConvert = decltype(convert_tag)::value;
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) bf16x4* lds_bf16x4_t;
    const uint8_t* cur = smem + (it & 1) * kStageBytes;
    uint8_t* nxt = smem + ((it + 1) & 1) * kStageBytes;
    const uint8_t* k_lane = cur + l32 * kKPitch + lh * 16;
    const uint8_t* v_lane = cur + 2 * kKTileBytes + (4 * lh + ((lane & 15) >> 2)) * kVPitch + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
    uint8_t* kdst = nxt + k_dst_off;
    uint8_t* vdst = nxt + v_dst_off;
    constexpr int kAhead = 5, kRing = 6;
    uint4 fk[kRing];
    bf16x4 fv[2][4][2];
    float16v sc[2][2];
    uint32_t pw[2][16];
    half2v s2[2], t[4];
    float v8[8], x[2][2], e[2][2];
    float neg = -m_run * p.scale_log2, sum = 0.0f;
    const float gs_k = k_gs, gs_v = v_gs;
    const uint8_t *values, *scales;  // where the raw registers are filled from next
    bool there;
    auto read_k = [&](auto tag) __attribute__((always_inline)) {  // fragment f % 16 of the 64 keys f / 16
      constexpr int f = decltype(tag)::value;
      fk[f % kRing] = *reinterpret_cast<const uint4*>(k_lane + (f >> 4) * kKTileBytes + ((f >> 3) & 1) * 32 * kKPitch + (f & 7) * 32);
    };
    // The tile's probabilities are there, none of them multiplied yet.
    auto follow_maximum = [&](float16v (&s)[2], uint32_t (&w)[16]) __attribute__((always_inline)) {
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(sum <= 128.0f)) != 0, 0)) {
        float mx = s[0][0];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kt][r]);
        mx = max_over_wave_halves(mx);
        const bool raise = (mx - m_run) * p.scale_log2 > kRescaleStep;
        if (__builtin_amdgcn_ballot_w64(raise) != 0) {
          const float alpha = raise ? __builtin_amdgcn_exp2f((m_run - mx) * p.scale_log2) : 1.0f;
          m_run = raise ? mx : m_run;
          neg = -m_run * p.scale_log2;
          l_run *= alpha;
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
          sum = 0.0f;
#pragma unroll
          for (int pair = 0; pair < 16; ++pair) {
            const float p0 = __builtin_amdgcn_exp2f(fmaf(s[pair >> 3][2 * (pair & 7)], p.scale_log2, neg));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(s[pair >> 3][2 * (pair & 7) + 1], p.scale_log2, neg));
            sum += p0 + p1;
            w[pair] = pack_bf16(p0, p1);
          }
        }
      }
      l_run += sum;
      sum = 0.0f;
    };
    each_index(read_k, std::make_integer_sequence<int, kAhead>{});
    __builtin_amdgcn_sched_barrier(0);
    auto one_slot = [&](auto slot_tag) __attribute__((always_inline)) {
      constexpr int slot = decltype(slot_tag)::value;
      // LDS reads: K five slots ahead of its MFMA, V four
      if constexpr (slot + kAhead < 32) read_k(std::integral_constant<int, slot + kAhead>{});
      if constexpr (slot >= 28 && slot < 60) {
        constexpr int u = slot - 28, step = (u >> 2) & 3, dt = u & 3;
#pragma unroll
        for (int j = 0; j < 2; ++j)
          fv[step & 1][dt][j] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (lds_bf16x4_t)(v_lane + (u >> 4) * kVTileBytes + (16 * step + 8 * j) * kVPitch + dt * 64));
      }
      __builtin_amdgcn_sched_barrier(0);
      // S^T of the first and the second 64 keys in slots 0-31 (32 keys after 32 keys), their O^T in slots 32-63
      if constexpr (slot < 32) {
        constexpr int h = slot >> 4, kt = (slot >> 3) & 1, ks = slot & 7;
        const float16v zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        sc[h][kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fk[slot % kRing]), qf[ks], ks == 0 ? zero : sc[h][kt], 0, 0, 0);
      } else {
        constexpr int u = slot - 32, h = u >> 4, step = (u >> 2) & 3, dt = u & 3;
        const bf16x4(&v)[2] = fv[step & 1][dt];
        const bf16x8 a = __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7);
        const bf16x8 b = __builtin_bit_cast(bf16x8, make_uint4(pw[h][4 * step], pw[h][4 * step + 1], pw[h][4 * step + 2], pw[h][4 * step + 3]));
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, o[dt], 0, 0, 0);
      }
      // probabilities: a pair's multiply-adds, exponentials, packing and sum in three slots in a row
      constexpr int kFirst[2] = {9, 29};
      constexpr int g = slot < kFirst[1] ? 0 : 1, i = slot - kFirst[g];
      if constexpr (i >= 2 && i < 18) {
        constexpr int pair = i - 2;
        pw[g][pair] = pack_bf16(e[pair & 1][0], e[pair & 1][1]);
        asm volatile("" : "+v"(pw[g][pair]));  // here, and not sunk behind the branch to the MFMA that reads it
        sum += e[pair & 1][0] + e[pair & 1][1];
      }
      if constexpr (i >= 1 && i < 17) {
        constexpr int pair = i - 1;
        e[pair & 1][0] = __builtin_amdgcn_exp2f(x[pair & 1][0]);
        e[pair & 1][1] = __builtin_amdgcn_exp2f(x[pair & 1][1]);
      }
      if constexpr (i >= 0 && i < 16) {
        constexpr int pair = i, kt = pair >> 3, r = 2 * (pair & 7);
        x[pair & 1][0] = fmaf(sc[g][kt][r], p.scale_log2, neg);
        x[pair & 1][1] = fmaf(sc[g][kt][r + 1], p.scale_log2, neg);
      }
      // conversion of the next tile: a dword's conversions, scaling, widening and packing in four slots in a row
      constexpr int kK = slot < 8 ? slot : slot >= 28 && slot < 36 ? slot - 20 : -1, kV = slot >= 47 && slot < 63 ? slot - 47 : -1;
      if constexpr (kConvert && (kK >= 0 || kV >= 0)) {
        constexpr bool is_k = kK >= 0;
        constexpr int piece = is_k ? kK : kV, j = piece >> 2;  // dword j of the row
        const KRaw& raw = is_k ? kf : vf;
        const uint32_t w = j == 0 ? raw.v.x : j == 1 ? raw.v.y : j == 2 ? raw.v.z : raw.v.w;
        const float gs = is_k ? gs_k : gs_v;
        if constexpr (piece == 0) block_scales_f16(raw.scales, s2);
        if constexpr ((piece & 3) == 0) {
          t[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0);
          t[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1);
          t[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2);
          t[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3);
        }
        if constexpr ((piece & 3) == 1) {
#pragma unroll
          for (int n = 0; n < 4; ++n) t[n] = t[n] * s2[j >> 1];
        }
        if constexpr ((piece & 3) == 2) {
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            v8[2 * n] = widen_mul_lo(t[n], gs);
            v8[2 * n + 1] = widen_mul_hi(t[n], gs);
          }
        }
        if constexpr ((piece & 3) == 3)
          reinterpret_cast<uint4*>(is_k ? kdst : vdst)[j] =
              make_uint4(pack_bf16(v8[0], v8[1]), pack_bf16(v8[2], v8[3]), pack_bf16(v8[4], v8[5]), pack_bf16(v8[6], v8[7]));
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (slot == 28 || slot == 47) {
        follow_maximum(sc[slot == 28 ? 0 : 1], pw[slot == 28 ? 0 : 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      // raw bytes of the iteration behind the next one, K and V each once its registers are free
      if constexpr (kConvert && slot == 9) {
        advance();
        there = it + 2 < seg_end && iter_base + k_local < n_cached;
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kConvert && (slot == 32 || slot == 58)) {
        const int from = there ? k_slot : 0;
        values = (slot == 32 ? tab.kv : tab.vv)[from];
        scales = (slot == 32 ? tab.ks : tab.vs)[from];
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kConvert && (slot == 37 || slot == 63)) {
        fetch_row(values, scales, there ? k_vo : 0u, there ? k_so : 0u, slot == 37 ? kf : vf);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    each_index(one_slot, std::make_integer_sequence<int, 64>{});
  };

  // prologue: the segment's first iteration into its stage, raw registers <- the second one
  fetch_next();
  if constexpr (!WIDE) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint8_t* patch = smem + ((seg_begin & 1) ^ 1) * kStageBytes + wave * kWaveQueries * kKPitch + l32 * kKPitch + lh * 16;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(patch + 32 * ks));
  }
  decode_any(seg_begin & 1);
  advance();
  if (seg_begin + 1 < seg_end) fetch_next();
  __syncthreads();
  // Every load issued so far (Q fragments, first tiles) has to have landed before the loop: otherwise the
  // compiler's wait-count bookkeeping carries them into the loop and makes the MFMA phase wait for the
  // prefetch loads it has just issued.  0x0F70 = vmcnt(0), other counters untouched.
  __builtin_amdgcn_s_waitcnt(0x0F70);

  // Iterations whose own 128 keys all exist and whose successor is all FP4 form a prefix of the key range;
  // they run the interleaved body: wide_iteration for 256-query tiles, and for 128-query tiles S^T (64 keys x 32 queries) = 16
  // MFMAs in eight steps of two, each step also converting one dword of the prefetched K row (even steps) or V row (odd
  // steps) into the other LDS stage.  The rest (the bf16 chunk, the tail) runs in a loop of its own, without conversion beside
  // the MFMAs.
  const int n_fast = min(n_cached / kIterKeys, seg_end) - 1;
  if (wave_idle) {
    // A wave without queries: the conversion of its rows, the same number of barriers, nothing else.
    for (; it < n_fast; ++it) {
      uint8_t* nxt = smem + ((it + 1) & 1) * kStageBytes;
      const bool has_next2 = it + 2 < seg_end;
      const uint32_t wk[4] = {kf.v.x, kf.v.y, kf.v.z, kf.v.w}, wv[4] = {vf.v.x, vf.v.y, vf.v.z, vf.v.w};
      half2v ks2[2], vs2[2];
      block_scales_f16(kf.scales, ks2);
      block_scales_f16(vf.scales, vs2);
      uint8_t* kdst = nxt + k_dst_off;
      uint8_t* vdst = nxt + v_dst_off;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v8[8];
        fp4x8_to_f32(wk[j], ks2[j >> 1], k_gs, v8);
        reinterpret_cast<uint4*>(kdst)[j] = make_uint4(pack_bf16(v8[0], v8[1]), pack_bf16(v8[2], v8[3]),
                                                       pack_bf16(v8[4], v8[5]), pack_bf16(v8[6], v8[7]));
        fp4x8_to_f32(wv[j], vs2[j >> 1], v_gs, v8);
        reinterpret_cast<uint4*>(vdst)[j] = make_uint4(pack_bf16(v8[0], v8[1]), pack_bf16(v8[2], v8[3]),
                                                       pack_bf16(v8[4], v8[5]), pack_bf16(v8[6], v8[7]));
      }
      advance();
      if (has_next2) fetch_next();
      __syncthreads();
    }
  }
  if constexpr (WIDE) {
    for (; it < n_fast; ++it) {
      wide_iteration(std::true_type{});
      __syncthreads();
    }
  }
  for (; !WIDE && it < n_fast; ++it) {
    const uint8_t* cur = smem + (it & 1) * kStageBytes;
    uint8_t* nxt = smem + ((it + 1) & 1) * kStageBytes;
    const bool has_next2 = it + 2 < seg_end;
    const uint32_t wk[4] = {kf.v.x, kf.v.y, kf.v.z, kf.v.w}, wv[4] = {vf.v.x, vf.v.y, vf.v.z, vf.v.w};
    half2v ks2[2], vs2[2];
    block_scales_f16(kf.scales, ks2);
    block_scales_f16(vf.scales, vs2);
    uint8_t* kdst = nxt + k_dst_off;
    uint8_t* vdst = nxt + v_dst_off;
    {
      float16v sc[2];
      const uint8_t* krow0 = cur + kp * kKTileBytes + l32 * kKPitch + lh * 16;
      const uint8_t* krow1 = krow0 + 32 * kKPitch;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[kt][i] = 0.0f;
      // K fragments two steps ahead of their MFMAs, three sets in rotation, held in place by scheduling barriers.
      uint4 fk[3][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        fk[ks][0] = *reinterpret_cast<const uint4*>(krow0 + ks * 32);
        fk[ks][1] = *reinterpret_cast<const uint4*>(krow1 + ks * 32);
      }
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        if (ks < 6) {
          fk[(ks + 2) % 3][0] = *reinterpret_cast<const uint4*>(krow0 + (ks + 2) * 32);
          fk[(ks + 2) % 3][1] = *reinterpret_cast<const uint4*>(krow1 + (ks + 2) * 32);
        }
        __builtin_amdgcn_sched_barrier(0);
        const bf16x8 fa0 = __builtin_bit_cast(bf16x8, fk[ks % 3][0]), fa1 = __builtin_bit_cast(bf16x8, fk[ks % 3][1]);
        sc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa0, qf[ks], sc[0], 0, 0, 0);
        sc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa1, qf[ks], sc[1], 0, 0, 0);
        // One dword (8 elements) of the prefetched rows at a time, K in the even steps, V in the odd ones.
        {
          const int j = ks >> 1;
          const bool is_k = (ks & 1) == 0;
          float v8[8];
          fp4x8_to_f32(is_k ? wk[j] : wv[j], is_k ? ks2[j >> 1] : vs2[j >> 1], is_k ? k_gs : v_gs, v8);
          reinterpret_cast<uint4*>(is_k ? kdst : vdst)[j] = make_uint4(pack_bf16(v8[0], v8[1]), pack_bf16(v8[2], v8[3]),
                                                                       pack_bf16(v8[4], v8[5]), pack_bf16(v8[6], v8[7]));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      advance();
      if (has_next2) fetch_next();
      softmax_pv(sc, cur + 2 * kKTileBytes + kp * kVTileBytes);
    }
    __syncthreads();
  }

  // The rows of a chunk tile reach LDS in pieces of 1 KB, one load of 64 x 16 bytes each: 34 of K, 36 of V, the rows' padding
  // included (its lanes fetch the row's last 16 bytes again).  Wave w takes pieces w, w + 8, w + 16, w + 24 of either and
  // one of the six behind them; here the source offsets of its lanes.  2640 queries x 24 heads over 13200 bf16 keys take
  // 407 us; with 32 loads of 4 bytes per lane and iteration (one row each), which cost 100 vector instructions for their
  // addresses, 437 us; with 10560 of the keys cached 422 instead of 429 us (measured in turn).
  constexpr int kKPieces = 2 * kKTileBytes / 1024, kVPieces = 2 * kVTileBytes / 1024;
  static_assert(kKPieces * 1024 == 2 * kKTileBytes && kVPieces * 1024 == 2 * kVTileBytes && kKPieces + kVPieces <= 72, "nine pieces per wave at most");
  const int chunk_wave = __builtin_amdgcn_readfirstlane(wave);
  uint32_t k_piece[4], v_piece[4];
  int piece_lane = lane;
  auto source = [&](uint32_t piece, uint32_t pitch) __attribute__((always_inline)) {
    const uint32_t at = piece * 1024u + piece_lane * 16u, row = at / pitch;
    return row * ((uint32_t)p.H * (kHeadDim * 2u)) + min(at - row * pitch, kHeadDim * 2u - 16u);
  };
  auto locate_pieces = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      k_piece[i] = source(chunk_wave + 8 * i, kKPitch);
      v_piece[i] = source(chunk_wave + 8 * i, kVPitch);
    }
  };
  if constexpr (WIDE) locate_pieces();

  // Plain body: the S phase without interleaved conversion, masking in the last tile, and the successor tile
  // decoded after the MFMAs (or, for the chunk's own bf16 tiles, brought in ahead of them).
  for (; it < seg_end; ++it) {
    const uint8_t* cur = smem + (it & 1) * kStageBytes;
    // A successor that lies wholly in the bf16 chunk is brought in ahead of the MFMAs, straight from global memory into
    // the other stage.
    const bool next_is_chunk = it + 1 < seg_end && iter_base >= n_cached && iter_base + kIterKeys <= Lk_i && p.H <= 65536;  // iter_base = first key of tile it + 1; 32-bit offsets inside a tile
    if (next_is_chunk) {
      const uint32_t dst = lds_address(smem + ((it + 1) & 1) * kStageBytes) + chunk_wave * 1024;
      const int64_t src_off = ((int64_t)(iter_base - n_cached) * p.H + head) * kHeadDim;
      const void *k_base = wave_uniform(p.k_new + src_off), *v_base = wave_uniform(p.v_new + src_off);
      if constexpr (!WIDE) {  // no registers to keep the offsets in: formed anew
        asm volatile("" : "+v"(piece_lane));
        locate_pieces();
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) load_to_lds_b128(k_piece[i], k_base, dst + i * 8192);
#pragma unroll
      for (int i = 0; i < 4; ++i) load_to_lds_b128(v_piece[i], v_base, dst + 2 * kKTileBytes + i * 8192);
      if (chunk_wave < kKPieces - 32) {
        load_to_lds_b128(source(32 + chunk_wave, kKPitch), k_base, dst + 32 * 1024);
      } else if (chunk_wave < kKPieces - 32 + kVPieces - 32) {
        load_to_lds_b128(source(64 - kKPieces + chunk_wave, kVPitch), v_base, dst + 2 * kKTileBytes + (64 - kKPieces) * 1024);
      }
    }
    // No key missing, and not the only such iteration of the segment, whose first tile has its probabilities formed twice: 2640
    // queries x 24 heads over 226 keys 21.1 us in the plain body, 21.8 in slots, over 256 19.95 and 19.9, over 512 27.35 and 26.65, 7040 x
    // 24 over 128 33.2 and 34.2, over 256 44.0 and 43.0, over 1024 105.7 and 99.7.
    const bool whole = WIDE && (it + 1) * kIterKeys <= Lk_i && min(seg_end, Lk_i / kIterKeys) - seg_begin > 1;
    if constexpr (WIDE) {
      if (whole && !wave_idle) wide_iteration(std::false_type{});
    }
#pragma unroll 1
    for (int h = whole ? kHalves : 0; h < kHalves; ++h) {
      const int tile = WIDE ? h : kp;
      const int tile_base = it * kIterKeys + tile * kTileKeys;
      if (tile_base >= Lk_i || wave_idle) break;
      float16v sc[2];
      const uint8_t* krow0 = cur + tile * kKTileBytes + l32 * kKPitch + lh * 16;
      const uint8_t* krow1 = krow0 + 32 * kKPitch;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[kt][i] = 0.0f;
      uint4 fk[3][2];  // K fragments two steps ahead, as in the loop above
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        fk[ks][0] = *reinterpret_cast<const uint4*>(krow0 + ks * 32);
        fk[ks][1] = *reinterpret_cast<const uint4*>(krow1 + ks * 32);
      }
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        if (ks < 6) {
          fk[(ks + 2) % 3][0] = *reinterpret_cast<const uint4*>(krow0 + (ks + 2) * 32);
          fk[(ks + 2) % 3][1] = *reinterpret_cast<const uint4*>(krow1 + (ks + 2) * 32);
        }
        __builtin_amdgcn_sched_barrier(0);
        sc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fk[ks % 3][0]), qf[ks], sc[0], 0, 0, 0);
        sc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fk[ks % 3][1]), qf[ks], sc[1], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (tile_base + kTileKeys > Lk_i) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = tile_base + kt * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
            if (key >= Lk_i) sc[kt][r] = -INFINITY;
          }
      }
      softmax_pv(sc, cur + 2 * kKTileBytes + tile * kVTileBytes);
    }
    if (next_is_chunk) {
      iter_base += kIterKeys;  // the slot bookkeeping of advance() has no use beyond the cache
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the rows have landed in LDS
    } else if (it + 1 < seg_end) {
      decode_any((it + 1) & 1);
      advance();
      if (it + 2 < seg_end) fetch_next();
    }
    __syncthreads();
  }

  l_run += __shfl_xor(l_run, 32, 64);  // row sums were per wave half so far
  {  // epilogue of the segment, with its own copies of the thread's coordinates (see fresh_thread_index)
  const auto& c = reread_params();
  const int tid = fresh_thread_index(), lane = tid & 63, wave = tid >> 6;
  const int qq = WIDE ? wave : (wave & 3), kp = WIDE ? 0 : (wave >> 2);
  if constexpr (WIDE) {
    // Every wave has seen its segment of the key range for its 32 queries.
    bool write_out = true;
    if (seg_begin != 0 || seg_end != n_iter) {
      // Part of a tile.  Whoever arrives last at a tile combines the parts; the others leave their state in a
      // record (two records per workgroup: one for the first tile it touches, one for the last) and count
      // their arrival.  The parts are combined from the end of the key range backwards whoever does it, so
      // the result does not depend on the order of arrival.  The workgroup that holds the last part is
      // normally also the last to arrive (the segments are walked backwards, see above): if a look at the
      // counter shows that, it goes on from its registers without writing a record.
      const uint32_t wg = group_number(c.d.G);
      const uint32_t split_tile = (uint32_t)tile_id - c.d.whole_rounds * c.d.G - c.d.extra;  // the tile's number among the split ones
      auto record_of = [&](uint32_t g) {
        return c.partials + (size_t)record_of_part(g, split_tile, division_of(c)) * (partial_bytes(kQueries) / sizeof(float)) +
               wave * (66 * 64) + lane;
      };
      uint32_t g_first, g_last;
      parts_of_tile(split_tile, division_of(c), g_first, g_last);
      const int others = (int)(g_last - g_first);
      if (tid == 0)
        tab.last_arrival = wg == g_last && __hip_atomic_load(c.arrivals + split_tile, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == others;
      __syncthreads();
      const bool from_registers = tab.last_arrival != 0;
      write_out = from_registers;
      if (!from_registers) {
        if (!wave_idle) {
          float* mine = record_of(wg);
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) store_shared_f32(mine + (dt * 16 + i) * 64, o[dt][i]);
          store_shared_f32(mine + 64 * 64, m_run);
          store_shared_f32(mine + 65 * 64, l_run);
        }
        // Every wave waits until its own record stores are complete (vmcnt(0): a write-through store is
        // acknowledged once it is visible device-wide) before it reaches the barrier; thread 0 counts the arrival
        // behind that barrier, so no workgroup can see the count without the whole record being in memory.
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        if (tid == 0)
          tab.last_arrival = __hip_atomic_fetch_add(c.arrivals + split_tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == others;
        __syncthreads();
        write_out = tab.last_arrival != 0;
      }
      if (write_out) {
        if (tid == 0) __hip_atomic_store(c.arrivals + split_tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
        if (!from_registers) {  // start from nothing; the first step below turns that into the last part exactly
          m_run = -INFINITY;
          l_run = 0.0f;
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
        }
        for (int g = (int)g_last - (from_registers ? 1 : 0); g >= (int)g_first && !wave_idle; --g) {
          const float* theirs = record_of((uint32_t)g);
          const float m1 = load_shared_f32(theirs + 64 * 64), l1 = load_shared_f32(theirs + 65 * 64);
          const float m = fmaxf(m_run, m1);
          const float a0 = (m_run == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((m_run - m) * p.scale_log2);
          const float a1 = (m1 == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((m1 - m) * p.scale_log2);
          l_run = l_run * a0 + l1 * a1;
          m_run = m;
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] = o[dt][i] * a0 + load_shared_f32(theirs + (dt * 16 + i) * 64) * a1;
        }
      }
    }
    if (write_out) {
      float out_max = 0.0f;
      const float inv_l = 1.0f / l_run;
      const int64_t first_query = (int64_t)qtile * kQueries + qq * kWaveQueries;
      write_rows<4>(o, inv_l, smem + wave * kWaveQueries * kKPitch, lane, c.out + (first_query * p.H + head) * kHeadDim, p.H,
                    (int)min(c.Lq - first_query, (int64_t)kWaveQueries), out_max);
      if (c.sink.parts) {
        out_max = wave_max(out_max);
        if (lane == 0) amax_sink_update(AmaxSink{c.sink.parts, c.sink.epoch, c.sink.epoch_offset}, (uint32_t)tile_id * 8 + wave, out_max);
      }
    }
  } else {
    // ---- The two waves of a group of queries leave each other two of their four 32-column groups in LDS; wave kp keeps
    // groups 2 kp and 2 kp + 1.
    float4* xo = reinterpret_cast<float4*>(smem);                     // [wave][8][64 lanes]
    float2* xml = reinterpret_cast<float2*>(smem + 8 * 8 * 64 * 16);  // [wave][64]
    constexpr int kMergeBytes = 8 * 8 * 64 * 16 + 8 * 64 * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float16v give = kp == 0 ? o[2 + (i >> 2)] : o[i >> 2];
      xo[(wave * 8 + i) * 64 + lane] = make_float4(give[4 * (i & 3)], give[4 * (i & 3) + 1], give[4 * (i & 3) + 2], give[4 * (i & 3) + 3]);
    }
    xml[wave * 64 + lane] = make_float2(m_run, l_run);
    __syncthreads();
    float16v own[2];
    {
      const float2 other = xml[(wave ^ 4) * 64 + lane];
      const float m0 = kp == 0 ? m_run : other.x, m1 = kp == 0 ? other.x : m_run;  // first and second half of the key range
      const float m = fmaxf(m0, m1);
      const float a0 = __builtin_amdgcn_exp2f((m0 - m) * p.scale_log2);
      const float a1 = (m1 == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f((m1 - m) * p.scale_log2);
      const float mine = kp == 0 ? a0 : a1, theirs = kp == 0 ? a1 : a0;
      l_run = (kp == 0 ? l_run : other.y) * a0 + (kp == 0 ? other.y : l_run) * a1;
      m_run = m;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float4 x = xo[((wave ^ 4) * 8 + i) * 64 + lane];
        const float xs[4] = {x.x, x.y, x.z, x.w};
        const float16v keep = kp == 0 ? o[i >> 2] : o[2 + (i >> 2)];
#pragma unroll
        for (int j = 0; j < 4; ++j) own[i >> 2][4 * (i & 3) + j] = keep[4 * (i & 3) + j] * mine + xs[j] * theirs;
      }
    }
    if (c.parts > 1) {
      // Part of a tile.  The workgroups of a tile each leave (O^T, reference point, row sum) in a record of their own and count
      // their arrival; the last to arrive adds the parts up, from the first to the last, four at a time, its own from its
      // registers at its place in that order - so the result does not depend on the order of arrival.  Stores and count are
      // ordered as above.  Bound by the latency of the exchange past the L2 (store, count, load: about 8 us of a launch in
      // all), hence 16-byte accesses with all of four parts in flight and no look at the counter ahead of the stores.
      constexpr uint32_t kRecordBytes = (uint32_t)partial_bytes(kQueries), kWaveBytes = kRecordBytes / 8;
      constexpr int kInFlight = 4;
      const int parts = (int)c.parts, part = (int)(group_number(c.d.G) - (uint32_t)tile_id * c.parts);
      const auto records = __builtin_amdgcn_make_buffer_rsrc(c.partials, 0, 0xFFFFFFFFu, 0x00027000u);
      const uint32_t first_record = (uint32_t)tile_id * c.parts * kRecordBytes;
      const uint32_t at_o = wave * kWaveBytes + lane * 16, at_ml = wave * kWaveBytes + 8 * 1024 + lane * 8;
      {
        const uint32_t rec = first_record + part * kRecordBytes;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float16v& v = own[i >> 2];
          store_shared_b128(records, at_o + i * 1024, rec, float4v{v[4 * (i & 3)], v[4 * (i & 3) + 1], v[4 * (i & 3) + 2], v[4 * (i & 3) + 3]});
        }
        store_shared_b64(records, at_ml, rec, float2v{m_run, l_run});
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __syncthreads();
      if (tid == 0)
        tab.last_arrival = __hip_atomic_fetch_add(c.arrivals + tile_id, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
      __syncthreads();
      if (tab.last_arrival == 0) break;
      if (tid == 0) __hip_atomic_store(c.arrivals + tile_id, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
      float16v sum[2];
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) sum[d][i] = 0.0f;
      float m = -INFINITY, l = 0.0f;
      for (int q0 = 0; q0 < parts; q0 += kInFlight) {
        float4v v[kInFlight][8];
        float2v ml[kInFlight];
#pragma unroll
        for (int j = 0; j < kInFlight; ++j) {  // behind the last part: the last again, which is not used
          const uint32_t rec = first_record + min(q0 + j, parts - 1) * kRecordBytes;
          ml[j] = load_shared_b64(records, at_ml, rec);
#pragma unroll
          for (int i = 0; i < 8; ++i) v[j][i] = load_shared_b128(records, at_o + i * 1024, rec);
        }
        float mj[kInFlight], m_new = m;
#pragma unroll
        for (int j = 0; j < kInFlight; ++j) {
          mj[j] = q0 + j >= parts ? -INFINITY : q0 + j == part ? m_run : ml[j][0];
          m_new = fmaxf(m_new, mj[j]);
        }
        const float a = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - m_new) * p.scale_log2);
        m = m_new;
        l *= a;
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) sum[d][i] *= a;
#pragma unroll
        for (int j = 0; j < kInFlight; ++j) {
          if (q0 + j >= parts) break;
          const bool mine = q0 + j == part;
          const float w = mj[j] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((mj[j] - m_new) * p.scale_log2);
          l += (mine ? l_run : ml[j][1]) * w;
#pragma unroll
          for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[d][i] += (mine ? own[d][i] : v[j][4 * d + (i >> 2)][i & 3]) * w;
        }
      }
      l_run = l;
#pragma unroll
      for (int d = 0; d < 2; ++d) own[d] = sum[d];
    }
    float out_max = 0.0f;
    const float inv_l = 1.0f / l_run;
    const int64_t first_query = (int64_t)qtile * kQueries + qq * kWaveQueries;
    write_rows<2>(own, inv_l, smem + kMergeBytes + wave * kWaveQueries * kKPitch, lane, c.out + (first_query * p.H + head) * kHeadDim + 64 * kp, p.H,
                  (int)min(c.Lq - first_query, (int64_t)kWaveQueries), out_max);
    if (c.sink.parts) {
      out_max = wave_max(out_max);
      if (lane == 0) amax_sink_update(AmaxSink{c.sink.parts, c.sink.epoch, c.sink.epoch_offset}, (uint32_t)tile_id * 8 + wave, out_max);
    }
  }
  }
  if constexpr (!WIDE) break;
  __syncthreads();  // the stages are free for the next segment
  }  // segments
}

// ----------------------------------------------------------------------------- short launches
// One head x 32 queries per workgroup, its keys dealt to W waves in tiles of 32 (wave w takes tiles w, w + W, ...).
// A launch of a few hundred queries gives the kernel above a few dozen tiles of 128 or 256 queries: most compute units
// idle, and every wave walks the whole key range or leaves 135 KB of partial results in device memory.  Here each wave
// has LDS rows, registers and a softmax of its own, nothing but the merge at the end needs a barrier, and the longest
// chain is (keys / 32 / W) tiles.  What it costs is the conversion of every K and V row once per 32 instead of
// 128 or 256 queries: short_kernel_waves (attention_split.h) says up to where that pays.
//
// The contraction over the head dimension may run in any order as long as Q and K agree: step ks of lane half lh
// covers elements 64 lh + 8 ks .. + 7, so the K operand of a cached row comes straight out of 32 packed bytes and four
// scale bytes of the lane's own, without LDS.  Rows of the chunk (bf16) are loaded four whole rows per instruction
// straight into LDS, as V always passes through it (its operand needs the transposing read).
//
// Bound by the issue of instructions: per tile 16 MFMAs beside about 600 others where the keys are cached and 230 where not,
// and by the LDS that the chunk's rows pass through.  us, with a 64-bit product per loaded row and a division per cached key /
// with 32-bit offsets that K and V share / with loads that need no registers and no stores to LDS: 368 queries x 16 heads over
// 1472 bf16 keys 15.6 / 14.4 / 12.6, 736 x 12 over 512 12.35 / 11.4 / 9.8, 192 x 2 over 2048 17.4 / 16.3 / 12.9, 736 x 12 over 736
// cached + 736 30.2 / 29.0 / 28.1, 368 x 16 over 1104 + 368 19.3 / 18.9 / 18.7 (the chunk's first K rows asked for ahead of
// the cached tiles: 19.1).  The tile kernels take 31.5 and 32.1 us for the first and the last.  Each wave loading Q for
// itself, 16 bytes of each of 32 rows at a time, and a merge in 4-byte accesses cost 1.2 and 1.4 more there, 5.5 instead of
// 4.9 for 192 x 2 over 16 keys (now 4.4).
constexpr int kShortKeys = 32;                                                // keys per wave tile
// A wave's K rows and V rows lie unpadded, as loads from memory straight into LDS write them: piece c of 16 bytes of row r at
// position c ^ swizzle(r), which spreads the 16 rows of a K read and the 4 of a transposing V read over all banks.
constexpr int kShortRow = 256, kShortRows = kShortKeys * kShortRow;
__device__ __forceinline__ int swizzle(int row) { return (row & 3) << 2 | ((row >> 2) & 3); }
constexpr int kShortRecord = 66 * 64;                                         // floats of a wave's result in the merge, 16-byte aligned
constexpr int kShortWaveBytes = kShortRecord * 4;                             // its K and V rows before that
constexpr int kShortQueries = kWaveQueries * kShortRow;                       // the queries, behind the waves' rows
template <int W>
constexpr size_t kShortLds = (size_t)W * kShortWaveBytes + kShortQueries + sizeof(SlotTable);
static_assert(2 * kShortRows <= kShortWaveBytes && kShortWaveBytes % 16 == 0, "the merge reuses the waves' rows");
static_assert(kShortLds<8> <= 160 * 1024 && 2 * kShortLds<4> <= 160 * 1024, "one workgroup of eight waves or two of four fit a unit");

// amdgpu_waves_per_eu: 256 registers per lane, two waves per SIMD (one workgroup of eight or two of four per CU)
// CACHED: there are cached keys.  The first tile's bytes are asked for with the queries (without cached keys) or as soon as
// the slot pointers are there (with them, the slots' scales still on their way), and a tile's rows without conditions,
// which the compiler turns into sixteen branches per tile (368 x 16 over 1472 16.1 instead of 14.8 us when that was found).
template <int W, bool CACHED>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void kv_attention_short_kernel(AttnParams p) {
  static_assert(W == 4 || W == 8, "the merge gives every wave 64 / W of the 64 output registers");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* const queries = smem + W * kShortWaveBytes;
  SlotTable& tab = *reinterpret_cast<SlotTable*>(queries + kShortQueries);
  float ka = 0.0f, va = 0.0f;
  if (const int t = threadIdx.x; CACHED && t < p.n_slots) {
    tab.kv[t] = reinterpret_cast<const uint8_t*>(p.kv_ptrs[t]);
    tab.ks[t] = reinterpret_cast<const uint8_t*>(p.ks_ptrs[t]);
    tab.vv[t] = reinterpret_cast<const uint8_t*>(p.vv_ptrs[t]);
    tab.vs[t] = reinterpret_cast<const uint8_t*>(p.vs_ptrs[t]);
    ka = load_global<float>(reinterpret_cast<const void*>(p.ka_ptrs[t]));
    va = load_global<float>(reinterpret_cast<const void*>(p.va_ptrs[t]));
  }
  const uint32_t tile_id = group_number(p.d.G);
  const int head = (int)(tile_id / (uint32_t)p.n_qtiles), qtile = (int)(tile_id - (uint32_t)head * (uint32_t)p.n_qtiles);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, lh = lane >> 5;
  const int n_cached = CACHED ? (int)p.n_cached : 0, n_new = (int)p.n_new;
  const int cached_tiles = (n_cached + kShortKeys - 1) / kShortKeys, n_tiles = cached_tiles + (n_new + kShortKeys - 1) / kShortKeys;
  uint8_t* const krows = smem + wave * kShortWaveBytes;
  uint8_t* const vrows = krows + kShortRows;
  int t = wave;

  // The chunk's own keys: piece j of a tile is rows 4 j + lane / 16, 16 bytes per lane.  Offsets of 32 bits for K and V alike: the
  // chunk has a few thousand keys (short_kernel_waves), and there are no more heads than twice the compute units.
  const uint32_t row_bytes = (uint32_t)p.H * kHeadDim * 2, last_row = (uint32_t)(n_new - 1) * row_bytes;
  const uint32_t krows_lds = lds_address(krows);
  const uint32_t piece = (uint32_t)((lane & 15) ^ (lane >> 4) << 2), column = (uint32_t)head * kHeadDim * 2;
  uint32_t at[8];
  auto fetch = [&](const uint16_t* src, uint32_t lds) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j) load_to_lds_b128(at[j], src, lds + j * 1024);
  };
  auto fetch_k = [&](int tile) __attribute__((always_inline)) {
    uint32_t first_row = (uint32_t)((tile - cached_tiles) * kShortKeys + (lane >> 4)) * row_bytes;
    asm volatile("" : "+v"(first_row));  // one running offset and not eight
#pragma unroll
    for (int j = 0; j < 8; ++j)  // behind the last key: the last again (V: zeros in LDS)
      at[j] = min(first_row + 4 * j * row_bytes, last_row) + ((piece ^ (j & 3)) * 16 + column);
    fetch(p.k_new, krows_lds);
  };
  auto fetch_v = [&]() __attribute__((always_inline)) { fetch(p.v_new, krows_lds + kShortRows); };  // of the tile of the last fetch_k
  // Cached keys: lane = (key l32, half lh of the head dimension) for K and V alike.
  struct { uint4 v[2]; uint32_t scales; } kf, vf;
  uint32_t slot = 0;
  // key / bts by a product: exact while key * bts < 2^31, and here both are a few thousand (short_kernel_waves)
  const uint32_t per_slot = CACHED ? (0x80000000u + (uint32_t)p.bts - 1u) / (uint32_t)p.bts : 0u;
  auto fetch_cached = [&](int tile) __attribute__((always_inline)) {
    const uint32_t key = (uint32_t)min(tile * kShortKeys + l32, n_cached - 1);
    slot = __umulhi(2u * key, per_slot);
    const int64_t row = (int64_t)(key - slot * (uint32_t)p.bts) * p.H + head;
    const uint32_t vo = (uint32_t)row * 64u + lh * 32u, so = (uint32_t)blocked_scale_offset(row, lh * 4, 8);
    kf.v[0] = load_global_b128(tab.kv[slot] + vo);
    kf.v[1] = load_global_b128(tab.kv[slot] + vo + 16);
    kf.scales = load_global<uint32_t>(tab.ks[slot] + so);
    vf.v[0] = load_global_b128(tab.vv[slot] + vo);
    vf.v[1] = load_global_b128(tab.vv[slot] + vo + 16);
    vf.scales = load_global<uint32_t>(tab.vs[slot] + so);
  };

  // piece 8 lh + i of row l32
  const uint32_t own_row0 = (uint32_t)(l32 * kShortRow + ((8 * lh) ^ swizzle(l32)) * 16);
  auto own_row = [&](int i) { return own_row0 ^ (uint32_t)(16 * i); };
  const int64_t query = (int64_t)qtile * kWaveQueries + l32;
  bf16x8 qf[8];
  {
    // The waves bring the queries into LDS together, 32 / W rows each, four rows per load, and all read the same fragments.
#pragma unroll
    for (int it = 0; it < 8 / W; ++it) {
      const int group = wave * (8 / W) + it;
      const uint32_t row = (uint32_t)min((int64_t)qtile * kWaveQueries + group * 4 + (lane >> 4), p.Lq - 1);
      load_to_lds_b128(row * row_bytes + (piece ^ (uint32_t)(group & 3)) * 16 + column, p.q, lds_address(queries) + group * 1024);
    }
    if (!CACHED) {  // a wave without a tile loads the last
      fetch_k(min(t, n_tiles - 1));
      fetch_v();
    }
    if (CACHED) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(16)" ::: "memory");  // K and V of the first tile
    __syncthreads();  // and the slot pointers
    if (CACHED && (int)threadIdx.x < p.n_slots) {
      tab.kg[threadIdx.x] = ka * p.inv_denom;
      tab.vg[threadIdx.x] = va * p.inv_denom;
    }
    if (CACHED && t < cached_tiles) fetch_cached(t);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(queries + own_row(ks)));
  }
  if (CACHED) __syncthreads();  // the slots' scales

  float16v o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;
  float neg = 0.0f;  // the reference point in the exponent of 2; 0 while no score above -inf has been met: all weigh nothing
  // The reference point follows the maximum in steps.  A probability close below its reference point loses least in bf16, and
  // the largest ones weigh most: with steps of 2^2, all queries of the wave raised as soon as one has to be, the result is
  // closer to fp64 than that of the divided tiles (368 queries x 16 heads over 1472 keys 0.00220 relative against 0.00224,
  // 192 x 2 over 960 0.00215 / 0.00219).  With the steps of 2^8 of the kernel above, which has larger tiles, it was further off
  // (0.00228, 0.00226).  The raises cost 1 to 2.5 % (368 x 16 over 1472 bf16 keys 17.5 -> 17.9 us).
  constexpr float kRescaleStep = 2.0f;

  // Softmax of the wave's 32 scores per query (register r of sc: key 8 (r / 4) + 4 lh + r % 4 of the tile, `valid` keys
  // exist) and O^T += V^T P^T from the V rows in LDS.
  // `v_there()`: the V rows are in LDS.
  // Row 4 lh + (lane / 4) % 4 + 8 j + 16 step of V, elements 32 dt + 16 (lane / 16 % 2) + 4 (lane % 4) .. + 3: with j, 16 step and dt.
  const uint32_t v_row0 = (uint32_t)((4 * lh + ((lane >> 2) & 3)) * kShortRow + (lane & 1) * 8);
  const uint32_t v_piece = (uint32_t)(((lane >> 2) & 3) << 2 | ((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ lh));
  auto softmax_pv = [&](float16v& sc, int valid, auto v_there) __attribute__((always_inline)) {
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) bf16x4* lds_bf16x4_t;
    bf16x4 vfr[2][4][2];
    auto read_v = [&](int step) __attribute__((always_inline)) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          vfr[step][dt][j] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (lds_bf16x4_t)(vrows + v_row0 + (16 * step + 8 * j) * kShortRow + (v_piece ^ (uint32_t)(4 * dt + 2 * j)) * 16));
    };
    if (valid < kShortKeys) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * lh + (r & 3) >= valid) sc[r] = -INFINITY;
    }
    float mx = sc[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sc[r]);
    mx = max_over_wave_halves(mx);
    if (__builtin_amdgcn_ballot_w64((mx - m_run) * p.scale_log2 > kRescaleStep) != 0) {
      const float m_new = fmaxf(m_run, mx);
      neg = m_new == -INFINITY ? 0.0f : -m_new * p.scale_log2;
      const float alpha = __builtin_amdgcn_exp2f(fmaf(m_run, p.scale_log2, neg));
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    v_there();
    read_v(0);
    read_v(1);
#pragma unroll
    for (int step = 0; step < 2; ++step) {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[8 * step + 2 * i], p.scale_log2, neg));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[8 * step + 2 * i + 1], p.scale_log2, neg));
        l_run += p0 + p1;
        w[i] = pack_bf16(p0, p1);
      }
      const bf16x8 pb = __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const bf16x8 a = __builtin_shufflevector(vfr[step][dt][0], vfr[step][dt][1], 0, 1, 2, 3, 4, 5, 6, 7);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pb, o[dt], 0, 0, 0);
      }
    }
    // the next tile's rows are written behind these reads: LDS accesses of one wave are carried out in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto rows_written = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  // ---- cached keys
  if constexpr (CACHED) {
    float kg = tab.kg[slot], vg = tab.vg[slot];
    for (; t < cached_tiles; t += W) {
      const int valid = n_cached - t * kShortKeys;
      float16v sc;
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[i] = 0.0f;
      const uint32_t wk[8] = {kf.v[0].x, kf.v[0].y, kf.v[0].z, kf.v[0].w, kf.v[1].x, kf.v[1].y, kf.v[1].z, kf.v[1].w};
      const bool live = l32 < valid;  // rows of keys that do not exist are zeros
      uint32_t wv[8] = {vf.v[0].x, vf.v[0].y, vf.v[0].z, vf.v[0].w, vf.v[1].x, vf.v[1].y, vf.v[1].z, vf.v[1].w};
#pragma unroll
      for (int j = 0; j < 8; ++j) wv[j] = live ? wv[j] : 0u;
      half2v ks2[4], vs2[4];
      block_scales_f16(kf.scales, *reinterpret_cast<half2v(*)[2]>(&ks2[0]));
      block_scales_f16(kf.scales >> 16, *reinterpret_cast<half2v(*)[2]>(&ks2[2]));
      const uint32_t vsc = live ? vf.scales : 0u;
      block_scales_f16(vsc, *reinterpret_cast<half2v(*)[2]>(&vs2[0]));
      block_scales_f16(vsc >> 16, *reinterpret_cast<half2v(*)[2]>(&vs2[2]));
      const float kgt = kg, vgt = live ? vg : 0.0f;
      if (t + W < cached_tiles) {
        fetch_cached(t + W);
        kg = tab.kg[slot];
        vg = tab.vg[slot];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float v8[8];
        fp4x8_to_f32(wk[j], ks2[j >> 1], kgt, v8);
        const bf16x8 fa = __builtin_bit_cast(bf16x8, make_uint4(pack_bf16(v8[0], v8[1]), pack_bf16(v8[2], v8[3]),
                                                                pack_bf16(v8[4], v8[5]), pack_bf16(v8[6], v8[7])));
        sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, qf[j], sc, 0, 0, 0);
        fp4x8_to_f32(wv[j], vs2[j >> 1], vgt, v8);
        *reinterpret_cast<uint4*>(vrows + own_row(j)) =
            make_uint4(pack_bf16(v8[0], v8[1]), pack_bf16(v8[2], v8[3]), pack_bf16(v8[4], v8[5]), pack_bf16(v8[6], v8[7]));
      }
      rows_written();
      softmax_pv(sc, valid, [] {});
    }
  }
  // ---- the chunk's own keys.  A tile's K rows are replaced by the next one's when they have been read, likewise its V rows, so
  // that either is under way while the other is worked on.
  if (t < n_tiles) {
    if (CACHED) {
      // The last cached tile's V rows are read: the loads that replace them are none that the compiler would wait ahead of.
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      fetch_k(t);
      fetch_v();
    }
    for (; t < n_tiles; t += W) {
      const int valid = n_new - (t - cached_tiles) * kShortKeys;
      const bool more = t + W < n_tiles;
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");  // K; V behind it
      float16v sc;
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[i] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
        sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(krows + own_row(ks))), qf[ks], sc, 0, 0, 0);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // all read
      if (more) fetch_k(t + W);
      softmax_pv(sc, valid, [&] {
        if (more) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (valid < kShortKeys) {  // nothing but zeros weighed with zero
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (4 * j + (lane >> 4) >= valid) *reinterpret_cast<uint4*>(vrows + j * 1024 + lane * 16) = make_uint4(0u, 0u, 0u, 0u);
          rows_written();
        }
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (more) fetch_v();
    }
  }

  // ---- merge: every wave leaves (O^T, reference point, row sum) where its rows were, wave w combines registers 64 w / W .. of
  // all.  Four registers per access: register 4 g + i of a lane is element i of its g-th group.
  l_run += __shfl_xor(l_run, 32, 64);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // a wave without a tile has loaded one all the same
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  auto record = [&](int w) { return reinterpret_cast<float*>(smem + w * kShortWaveBytes) + lane * 4; };
  {
    float* mine = record(wave);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(mine + (dt * 4 + g) * 256) = make_float4(o[dt][4 * g], o[dt][4 * g + 1], o[dt][4 * g + 2], o[dt][4 * g + 3]);
    *reinterpret_cast<float2*>(mine + 64 * 64 - 2 * lane) = make_float2(m_run, l_run);
  }
  __syncthreads();
  float a[W], m = -INFINITY, l = 0.0f;
  float2 ml[W];
#pragma unroll
  for (int w = 0; w < W; ++w) {
    ml[w] = *reinterpret_cast<const float2*>(record(w) + 64 * 64 - 2 * lane);
    m = fmaxf(m, ml[w].x);
  }
#pragma unroll
  for (int w = 0; w < W; ++w) {
    a[w] = ml[w].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((ml[w].x - m) * p.scale_log2);  // a wave without a tile: -inf
    l += a[w] * ml[w].y;
  }
  const float inv_l = 1.0f / l;
  float out_max = 0.0f;
#pragma unroll
  for (int g = 0; g < 16 / W; ++g) {
    const int reg = wave * (64 / W) + 4 * g;  // four registers = four neighbouring elements of the head dimension
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float4 x = *reinterpret_cast<const float4*>(record(w) + (reg >> 2) * 256);
      v[0] += a[w] * x.x;
      v[1] += a[w] * x.y;
      v[2] += a[w] * x.z;
      v[3] += a[w] * x.w;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= inv_l;
    if (query < p.Lq) {
      const uint2 packed = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
      const int d = 32 * (reg >> 4) + 8 * ((reg & 15) >> 2) + 4 * lh;
      *reinterpret_cast<uint2*>(p.out + (query * p.H + head) * kHeadDim + d) = packed;
      out_max = abs_max_bf16x8(make_uint4(packed.x, packed.y, 0u, 0u), out_max);
    }
  }
  if (p.sink.parts) {
    out_max = wave_max(out_max);
    if (lane == 0) amax_sink_update(p.sink, tile_id * W + wave, out_max);
  }
}

static std::atomic<int> g_attention_policy{LL_ATTENTION_AUTO};

// Short launches take kv_attention_short_kernel, under the automatic choice and where the division without shared tiles and
// with few queries per workgroup (LL_ATTENTION_NARROW) is asked for.  For the others there are four ways, all one workgroup
// per compute unit at a time (LDS):
//  * 128 queries per workgroup, the key range halved between two sets of waves; one workgroup per tile;
//  * 256 queries per workgroup (every decoded K/V tile serves twice as many MFMAs: an iteration takes about 1.64
//    times as long for twice the work), one workgroup per tile;
//  * 256 queries per workgroup, whole rounds of tiles first and the (tile, iteration) sequence of the tiles behind
//    them cut into one equal share per compute unit; tiles that straddle two shares are combined by the workgroup
//    that finishes last;
//  * 128 queries per workgroup where there are few tiles: the same number of workgroups share the key range of each, all
//    of them in one round, combined likewise.
// plan_division (attention_split.h) chooses: plan_attention among the first three, then between that and the fourth.
static int launch_attention(const AttnParams& p_in, hipStream_t stream) {
  AttnParams p = p_in;
  const size_t smem = 2 * kStageBytes + sizeof(SlotTable);
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    set_error("ll_kv_attention: hipGetDevice failed");
    return LL_ELAUNCH;
  }
  if (int rc = compute_units_of(dev, cus, "ll_kv_attention")) return rc;
  const int64_t n_iter = (p.n_cached + p.n_new + kIterKeys - 1) / kIterKeys;
  LL_REQUIRE(p.H * ((p.Lq + kWgQueries - 1) / kWgQueries) * n_iter < (1ll << 32), "ll_kv_attention: too many (tile, iteration) units");
  const int policy = g_attention_policy.load(std::memory_order_relaxed);
  if (const int waves = short_kernel_waves(p.Lq, p.H, p.n_cached, p.n_new, cus, policy)) {
    p.n_qtiles = (int)((p.Lq + kWaveQueries - 1) / kWaveQueries);
    p.d.G = (uint32_t)(p.H * p.n_qtiles);
    static std::atomic<uint64_t> lds_allowed[4] = {};
#define LL_LAUNCH_SHORT(W, CACHED, i)                                                                                      \
  const void* kernel = reinterpret_cast<const void*>(&kv_attention_short_kernel<W, CACHED>);                               \
  if (int rc = allow_dynamic_lds(kernel, kShortLds<W>, lds_allowed[i], "ll_kv_attention")) return rc;                      \
  hipLaunchKernelGGL((kv_attention_short_kernel<W, CACHED>), dim3(p.d.G), dim3(W * 64), kShortLds<W>, stream, p)
    if (waves == 8 && p.n_cached > 0) {
      LL_LAUNCH_SHORT(8, true, 0);
    } else if (waves == 8) {
      LL_LAUNCH_SHORT(8, false, 1);
    } else if (p.n_cached > 0) {
      LL_LAUNCH_SHORT(4, true, 2);
    } else {
      LL_LAUNCH_SHORT(4, false, 3);
    }
#undef LL_LAUNCH_SHORT
    LL_CHECK_LAUNCH("kv_attention_short_kernel");
    return LL_OK;
  }
  AttentionPlan plan = plan_division(p.Lq, p.H, p.n_cached, p.n_new, cus, policy);
  StreamScratch w;
  if (plan.mode == LL_ATTENTION_SPLIT) {
    // The split division passes partial tiles through device memory of the library's own.  While the stream is
    // being captured nothing may be allocated (and the clearing of a new set must not become a graph node): a set
    // that an earlier launch or ll_kv_attention_reserve left on this stream is used as it is; without one the
    // automatic choice falls back to the cheaper of the two divisions that need no memory, and an explicit
    // request for the split division is refused.
    bool missing = false;
    if (int rc = stream_scratch(dev, stream, partial_records(plan) * partial_bytes(plan.queries), (size_t)plan.split_tiles,
                                !stream_is_capturing(stream), w, &missing, "ll_kv_attention")) return rc;
    if (missing) {
      if (policy == LL_ATTENTION_SPLIT) {
        set_error("ll_kv_attention: the split division needs device memory that cannot be allocated while the stream "
                  "is being captured; call ll_kv_attention_reserve for this shape first, or select another division");
        return LL_ENOSUP;
      }
      plan = plan_attention(p.Lq, p.H, p.n_cached + p.n_new, cus, policy, /*allow_split=*/false);
    }
  }
  p.n_qtiles = plan.n_qtiles;
  p.full_qtiles = plan.full_qtiles;
  p.d = plan.d;
  p.parts = (uint32_t)plan.parts;
  if (plan.mode == LL_ATTENTION_SPLIT) {
    p.partials = reinterpret_cast<float*>(w.records);
    p.arrivals = w.counters;
  }
  if (plan.queries == kWgQueries) {
    static std::atomic<uint64_t> lds_allowed{0};
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&kv_attention_kernel<false>), smem, lds_allowed, "ll_kv_attention")) return rc;
    hipLaunchKernelGGL(kv_attention_kernel<false>, dim3(p.d.G), dim3(kAttnThreads), smem, stream, p);
  } else {
    static std::atomic<uint64_t> lds_allowed_w{0};
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&kv_attention_kernel<true>), smem, lds_allowed_w, "ll_kv_attention")) return rc;
    hipLaunchKernelGGL(kv_attention_kernel<true>, dim3(p.d.G), dim3(kAttnThreads), smem, stream, p);
  }
  LL_CHECK_LAUNCH("kv_attention_kernel");
  return LL_OK;
}

}  // namespace ll

extern "C" int ll_kv_attention_set_policy(int policy) {
  LL_REQUIRE(policy >= LL_ATTENTION_AUTO && policy <= LL_ATTENTION_SPLIT, "ll_kv_attention_set_policy: unknown policy %d", policy);
  ll::g_attention_policy.store(policy);
  return LL_OK;
}

extern "C" int ll_kv_attention_get_policy(void) { return ll::g_attention_policy.load(); }

extern "C" int ll_kv_attention_reserve_window(int64_t Lq, int num_heads, int64_t n_cached, int64_t n_new, void* stream) {
  using namespace ll;
  LL_REQUIRE(Lq > 0 && num_heads > 0 && n_cached >= 0 && n_new >= 0 && n_cached + n_new > 0 && Lq < (1ll << 30) && n_cached < (1ll << 30) &&
                 n_new < (1ll << 30) && n_cached + n_new < (1ll << 30),
             "ll_kv_attention_reserve: bad sizes");
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    set_error("ll_kv_attention_reserve: hipGetDevice failed");
    return LL_ELAUNCH;
  }
  if (int rc = compute_units_of(dev, cus, "ll_kv_attention")) return rc;
  const int policy = g_attention_policy.load(std::memory_order_relaxed);
  if (short_kernel_waves(Lq, num_heads, n_cached, n_new, cus, policy)) return LL_OK;
  const AttentionPlan plan = plan_division(Lq, num_heads, n_cached, n_new, cus, policy);
  if (plan.mode != LL_ATTENTION_SPLIT) return LL_OK;
  if (stream_is_capturing(static_cast<hipStream_t>(stream))) {
    set_error("ll_kv_attention_reserve: the stream is being captured; reserve before the recording starts");
    return LL_ENOSUP;
  }
  StreamScratch w;
  return stream_scratch(dev, static_cast<hipStream_t>(stream), partial_records(plan) * partial_bytes(plan.queries),
                        (size_t)plan.split_tiles, true, w, nullptr, "ll_kv_attention_reserve");
}

// Cached keys are the longer way through the short kernel, and one fresh key may make a tile more: where these two need no
// memory, no other division of the keys into cached and fresh ones does.
extern "C" int ll_kv_attention_reserve(int64_t Lq, int num_heads, int64_t n_keys, void* stream) {
  if (int rc = ll_kv_attention_reserve_window(Lq, num_heads, n_keys, 0, stream)) return rc;
  return n_keys > 1 ? ll_kv_attention_reserve_window(Lq, num_heads, n_keys - 1, 1, stream) : LL_OK;
}

extern "C" int ll_kv_attention_release(void* stream) { return ll_release_stream_memory(stream); }

extern "C" int ll_kv_attention_plan_window(int64_t Lq, int num_heads, int64_t n_cached, int64_t n_new, int compute_units, int policy,
                                           int* division, uint32_t* workgroups, uint32_t* whole_rounds, int64_t* split_tiles) {
  LL_REQUIRE(Lq > 0 && num_heads > 0 && n_cached >= 0 && n_new >= 0 && n_cached + n_new > 0 && compute_units > 0 && Lq < (1ll << 30) &&
                 n_cached < (1ll << 30) && n_new < (1ll << 30) && n_cached + n_new < (1ll << 30),
             "ll_kv_attention_plan: bad sizes");
  LL_REQUIRE(policy >= LL_ATTENTION_AUTO && policy <= LL_ATTENTION_SPLIT, "ll_kv_attention_plan: unknown policy %d", policy);
  if (ll::short_kernel_waves(Lq, num_heads, n_cached, n_new, compute_units, policy)) {
    if (division) *division = LL_ATTENTION_NARROW;
    if (workgroups) *workgroups = (uint32_t)(num_heads * ((Lq + 31) / 32));
    if (whole_rounds) *whole_rounds = 1;
    if (split_tiles) *split_tiles = 0;
    return LL_OK;
  }
  const ll::AttentionPlan plan = ll::plan_division(Lq, num_heads, n_cached, n_new, compute_units, policy);
  if (division) *division = plan.mode;
  if (workgroups) *workgroups = plan.d.G;
  if (whole_rounds) *whole_rounds = plan.d.whole_rounds;
  if (split_tiles) *split_tiles = plan.split_tiles;
  return LL_OK;
}

extern "C" int ll_kv_attention_plan(int64_t Lq, int num_heads, int64_t n_keys, int compute_units, int policy,
                                    int* division, uint32_t* workgroups, uint32_t* whole_rounds, int64_t* split_tiles) {
  return ll_kv_attention_plan_window(Lq, num_heads, 0, n_keys, compute_units, policy, division, workgroups, whole_rounds, split_tiles);
}

extern "C" int ll_kv_attention(const void* q, int64_t Lq, int num_heads, const uint64_t* k_values_ptrs,
                               const uint64_t* k_scales_ptrs, const uint64_t* k_amax_ptrs,
                               const uint64_t* v_values_ptrs, const uint64_t* v_scales_ptrs,
                               const uint64_t* v_amax_ptrs, int64_t n_cached, int block_token_size, float e2m1_max,
                               float e4m3_max, const void* k_new, const void* v_new, int64_t n_new,
                               float softmax_scale, void* out, void* stream) {
  return ll_kv_attention_amax(q, Lq, num_heads, k_values_ptrs, k_scales_ptrs, k_amax_ptrs, v_values_ptrs,
                              v_scales_ptrs, v_amax_ptrs, n_cached, block_token_size, e2m1_max, e4m3_max, k_new, v_new,
                              n_new, softmax_scale, out, nullptr, stream);
}

extern "C" int ll_kv_attention_amax(const void* q, int64_t Lq, int num_heads, const uint64_t* k_values_ptrs,
                                    const uint64_t* k_scales_ptrs, const uint64_t* k_amax_ptrs,
                                    const uint64_t* v_values_ptrs, const uint64_t* v_scales_ptrs,
                                    const uint64_t* v_amax_ptrs, int64_t n_cached, int block_token_size,
                                    float e2m1_max, float e4m3_max, const void* k_new, const void* v_new,
                                    int64_t n_new, float softmax_scale, void* out, const ll_amax_sink* amax_sink,
                                    void* stream) {
  using namespace ll;
  LL_REQUIRE(q && out, "ll_kv_attention: null q/out");
  LL_REQUIRE(Lq > 0 && num_heads > 0 && n_cached >= 0 && n_new >= 0 && n_cached + n_new > 0,
             "ll_kv_attention: bad sizes Lq=%lld H=%d n_cached=%lld n_new=%lld", (long long)Lq, num_heads,
             (long long)n_cached, (long long)n_new);
  LL_REQUIRE(n_new == 0 || (k_new && v_new), "ll_kv_attention: n_new > 0 needs k_new and v_new");
  LL_REQUIRE(n_cached + n_new < (1ll << 30) && Lq < (1ll << 30), "ll_kv_attention: sequence too long");
  int n_slots = 0;
  if (n_cached > 0) {
    LL_REQUIRE(k_values_ptrs && k_scales_ptrs && k_amax_ptrs && v_values_ptrs && v_scales_ptrs && v_amax_ptrs,
               "ll_kv_attention: n_cached > 0 needs the six slot pointer tables");
    LL_REQUIRE(block_token_size >= 4 && e2m1_max > 0.f && e4m3_max > 0.f, "ll_kv_attention: bad slot geometry");
    LL_REQUIRE((int64_t)block_token_size * num_heads * 64 < (1ll << 31), "ll_kv_attention: slot too large");
    LL_REQUIRE(((int64_t)block_token_size * num_heads) % 128 == 0,
               "ll_kv_attention: slot rows (block_token_size*num_heads = %lld) must be a multiple of 128",
               (long long)block_token_size * num_heads);
    n_slots = (int)((n_cached + block_token_size - 1) / block_token_size);
    LL_REQUIRE(n_slots <= kMaxSlots, "ll_kv_attention: at most %d cache slots, got %d", kMaxSlots, n_slots);
  }
  LL_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(k_new) |
               reinterpret_cast<uintptr_t>(v_new)) & 15) == 0,
             "ll_kv_attention: q, out, k_new, v_new must be 16-byte aligned");
  AttnParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.Lq = Lq;
  p.H = num_heads;
  p.kv_ptrs = k_values_ptrs; p.ks_ptrs = k_scales_ptrs; p.ka_ptrs = k_amax_ptrs;
  p.vv_ptrs = v_values_ptrs; p.vs_ptrs = v_scales_ptrs; p.va_ptrs = v_amax_ptrs;
  p.n_cached = n_cached;
  p.n_new = n_new;
  p.bts = n_cached > 0 ? block_token_size : (1 << 30);
  p.n_slots = n_slots;
  p.inv_denom = n_cached > 0 ? kv_inverse_denominator(e2m1_max, e4m3_max) : 0.f;
  p.k_new = static_cast<const uint16_t*>(k_new);
  p.v_new = static_cast<const uint16_t*>(v_new);
  p.scale_log2 = softmax_scale * 1.4426950408889634f;
  p.out = static_cast<uint16_t*>(out);
  LL_REQUIRE(sink_is_valid(amax_sink), "ll_kv_attention_amax: amax sink needs 8-byte alignment and a non-zero epoch");
  p.sink = make_sink(amax_sink);
  return launch_attention(p, static_cast<hipStream_t>(stream));
}

extern "C" int ll_attention_bf16(const void* q, const void* k, const void* v, int64_t Lq, int64_t Lk, int num_heads,
                                 float softmax_scale, void* out, void* stream) {
  return ll_kv_attention(q, Lq, num_heads, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 6.f, 256.f, k,
                         v, Lk, softmax_scale, out, stream);
}
