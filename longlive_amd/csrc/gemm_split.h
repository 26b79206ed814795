// How the persistent W4A4 GEMM divides a launch between its workgroups: the arithmetic shared by the kernel (device),
// the launcher (host) and the host-side checks of the test suite.  Integer arithmetic on four launch-wide numbers,
// identical on both sides.
//
// A launch has `tiles` output tiles (128 rows x 512 columns) of `nk` K steps (128 K elements) each and G workgroups.
// Workgroup g first runs `whole_rounds` whole tiles (tile j * G + g in round j): the workgroups of a round start
// together and move through K together, so those that share an XCD find each other's A and B lines in its L2.  The
// tiles behind the whole rounds, numbered from 0 as "split tiles", are cut into units (split tile t, step k is unit
// t * nk + k), and workgroup g takes the units [g * units / G, (g + 1) * units / G): at most the tail of one tile,
// whole tiles, and the head of another, walked from the end backwards one segment (a run of steps of one tile) at a
// time.  A segment that is not a whole tile leaves its fp32 partial tile in a record; the workgroup that arrives
// last at a tile adds the parts up, always in the same order, and writes the output.
#pragma once
#include <stdint.h>

#ifndef __HIPCC__
#define LL_GEMM_SPLIT_FN inline
#else
#define LL_GEMM_SPLIT_FN __host__ __device__ __forceinline__
#endif

namespace ll {

struct GemmDivision {
  uint32_t G;             // workgroups
  uint32_t tiles;         // output tiles
  uint32_t nk;            // K steps per tile
  uint32_t whole_rounds;  // whole tiles every workgroup runs first
};

LL_GEMM_SPLIT_FN uint32_t gemm_split_tiles(const GemmDivision& d) { return d.tiles - d.whole_rounds * d.G; }
LL_GEMM_SPLIT_FN uint64_t gemm_units(const GemmDivision& d) { return (uint64_t)gemm_split_tiles(d) * d.nk; }

// First unit of workgroup g's share (g = G: one past the last unit).
LL_GEMM_SPLIT_FN uint64_t gemm_first_unit(uint32_t g, const GemmDivision& d) { return (uint64_t)g * gemm_units(d) / d.G; }

// The workgroup whose share holds unit u: the g with first_unit(g) <= u < first_unit(g + 1).
LL_GEMM_SPLIT_FN uint32_t gemm_holder_of_unit(uint64_t u, const GemmDivision& d) {
  return (uint32_t)(((u + 1) * d.G - 1) / gemm_units(d));
}

struct GemmSegment {
  uint32_t tile;        // tile number in the launch (whole rounds first, split tiles behind them)
  uint32_t begin, end;  // K steps [begin, end) of the tile
};

// Position of a workgroup in its work: whole tiles done, and the end of what is left of its share of the units.
struct GemmCursor {
  uint32_t round;
  uint64_t share_end;
};

LL_GEMM_SPLIT_FN GemmCursor gemm_start_of_work(uint32_t g, const GemmDivision& d) {
  return GemmCursor{0u, gemm_units(d) ? gemm_first_unit(g + 1, d) : 0u};
}

// The next segment of workgroup g, or false when its work is done.
LL_GEMM_SPLIT_FN bool gemm_next_segment(GemmCursor& at, uint32_t g, const GemmDivision& d, GemmSegment& seg) {
  if (at.round < d.whole_rounds) {
    seg.tile = at.round * d.G + g;
    seg.begin = 0;
    seg.end = d.nk;
    ++at.round;
    return true;
  }
  if (gemm_units(d) == 0) return false;
  const uint64_t share_begin = gemm_first_unit(g, d);
  if (at.share_end <= share_begin) return false;
  const uint64_t split_tile = (at.share_end - 1) / d.nk, first = split_tile * d.nk;
  seg.tile = d.whole_rounds * d.G + (uint32_t)split_tile;
  seg.begin = share_begin > first ? (uint32_t)(share_begin - first) : 0u;
  seg.end = (uint32_t)(at.share_end - first);
  at.share_end = first + seg.begin;
  return true;
}

// The workgroups that hold a part of split tile `split_tile`: g_first .. g_last, every one of them.
LL_GEMM_SPLIT_FN void gemm_parts_of_tile(uint32_t split_tile, const GemmDivision& d, uint32_t& g_first, uint32_t& g_last) {
  g_first = gemm_holder_of_unit((uint64_t)split_tile * d.nk, d);
  g_last = gemm_holder_of_unit((uint64_t)split_tile * d.nk + d.nk - 1, d);
}

// Which of its two records workgroup g uses for its part of `split_tile`: the first one for the first tile its
// share touches, the second one otherwise (only the first and the last tile of a share can be partial).
LL_GEMM_SPLIT_FN uint32_t gemm_record_of_part(uint32_t g, uint32_t split_tile, const GemmDivision& d) {
  return 2 * g + ((uint32_t)(gemm_first_unit(g, d) / d.nk) == split_tile ? 0u : 1u);
}

// ---- the launcher's choice (host)
constexpr int kPTileM = 128, kPTileN = 512;  // rows and columns of an output tile

// Whether a launch runs the persistent kernel, and its division.
struct PersistentPlan {
  bool use;
  GemmDivision d;
  int tiles_m, tiles_n_each;
};
inline PersistentPlan plan_persistent(int64_t M, int64_t N, int64_t Kp, int n_products, int cus, int schedule) {
  PersistentPlan plan{};
  if (schedule == 0 /* LL_GEMM_TILES */ || schedule == 2 /* LL_GEMM_TILES_COMPILED */ || Kp % 128 != 0 || Kp >= (1 << 28) || cus < 1) return plan;
  const int64_t tiles_m = (M + kPTileM - 1) / kPTileM, tiles_n_each = (N + kPTileN - 1) / kPTileN;
  const int64_t tiles = tiles_m * tiles_n_each * n_products, nk = Kp / 128;
  if (tiles >= (1ll << 30) || tiles * nk < cus) return plan;
  // The automatic choice never takes the persistent launch.  One wave per SIMD has nobody to hide a tile's first
  // loads and its epilogue behind, and the tiles behind the whole rounds pay for their partial tiles: inside the DiT
  // block, with bias, GELU or the gated residual in the epilogue, every product measured slower (FFN-down 243 against
  // 221 us, FFN-up 300 against 224 us), and where it used to win alone (long K, at least a whole tile per workgroup:
  // 7040 x 3072 x 14336 in 505 us, 4096 x 4096 x 14336 in 355 us) the hand-scheduled tile kernels have caught up
  // (483 and 359 us).
  if (schedule == -1 /* LL_GEMM_AUTO */) return plan;
  int64_t rounds = tiles / cus;
  // A few left-over tiles would be cut into many thin parts each (or leave workgroups without a single K step, and
  // every workgroup of [first, last] must hold a part of a split tile): then one whole round joins the split part.
  if (const int64_t left = tiles % cus; left > 0 && rounds > 0 && (left * 8 < cus || left * nk < cus)) --rounds;
  plan.use = true;
  plan.d = GemmDivision{(uint32_t)cus, (uint32_t)tiles, (uint32_t)nk, (uint32_t)rounds};
  plan.tiles_m = (int)tiles_m;
  plan.tiles_n_each = (int)tiles_n_each;
  return plan;
}

// Which kernel runs the 64 x 64 tiles (LL_GEMM_KERNEL_64X64): gemm_w4a4_small_kernel from three K steps of 256 on, else the tile
// kernel, which has less to do before the first step and behind the last.  us, small kernel / tile kernel, by K:
//   tiles       64           256          512          768          1024         1536
//     8     4.4 / 3.6    4.3 / 4.1    4.9 / 5.0    5.4 / 6.0    6.1 / 7.0    7.2 / 8.9
//    72     4.5 / 3.5    4.4 / 4.0    5.0 / 4.9    5.5 / 5.9    6.2 / 6.9    7.3 / 8.8
//   384     5.4 / 4.5    5.3 / 5.4    6.5 / 6.7    7.3 / 8.2    8.2 / 9.7    10.0 / 12.7
// It addresses eight rows of Kp / 2 bytes with 32-bit offsets.
inline bool small_kernel_takes(int64_t Kp, int schedule) { return Kp > 512 && Kp < (1 << 28) && schedule != 2 /* LL_GEMM_TILES_COMPILED */; }

// ---- which one-workgroup-per-tile kernel a launch takes (host arithmetic; the values are the header's
// LL_GEMM_KERNEL_* codes)
struct TileKernelChoice {
  int kernel;           // 0: 64 x 64, 1: 128 x 128, 2: 128 x 256, 3: 256 x 128 (four waves); 4: 128 x 256, eight waves
  bool hand_scheduled;  // the generated main loop
};
inline TileKernelChoice choose_tile_kernel(int64_t M, int64_t N, int64_t Kp, int n_products, int cus, int schedule) {
  // the generated loops address a row band with 32-bit offsets: 16 rows of Kp / 2 bytes
  const int64_t tiles_64 = ((M + 63) / 64) * ((N + 63) / 64) * n_products;
  const bool generated_ok = Kp % 128 == 0 && Kp < (1 << 28) && schedule != 2 /* LL_GEMM_TILES_COMPILED */;
  // At most one 128 x 256 tile per compute unit, and more than half of the units busy: one workgroup of eight waves
  // per tile, the K range of every step split between its two halves.
  if (generated_ok && Kp >= 512) {
    const int64_t tiles = ((M + 127) / 128) * ((N + 255) / 256) * n_products;
    // ... unless the 64 x 64 tiles of the small-product kernel are no more than four and a half per unit: 1320 x 3072 x
    // 3072, 1008 of them: 28.5 against 36.8 us; x 768 12.8 / 14.9, x 14336 116 / 139; 1400 x 3072 x 3072, 1056: 34.8 /
    // 36.7; 1760 x 2560 x 2560, 1120: 30.0 / 32.3; but 736 x 8960 x 1536, 1680: 28.6 / 23.9.
    if (tiles <= cus && 2 * tiles > cus) {
      if (small_kernel_takes(Kp, schedule) && 2 * tiles_64 <= 9 * (int64_t)cus) return {0, false};
      return {4, true};
    }
  }
  // Small problems: when even 128 x 128 tiles would occupy at most half of the compute units, 64 x 64 tiles (more decode
  // work per MFMA, but four times the workgroups) finish sooner.  Up to three of them per unit they still do in the
  // small-product kernel, since each 128 x 128 tile then has a unit to itself or shares it with one other (us, that kernel
  // / tiles of 128 x 128): 1320 x 1536 x 1536, 504 small tiles: 10.4 / 16.1; x 640 7.5 / 9.2; 335 x 5888 x 1536, 552: 14.7
  // / 15.9; 1500 x 2048 x 1536, 768: 15.0 / 16.4; 1760 x 1536 x 768, 672: 10.3 / 10.3; but 2640 x 1024 x 640, 672: 10.4 /
  // 9.6; 736 x 4608 x 1536, 864: 18.2 / 16.5; 2048 x 2048 x 8192, 1024: 72.9 / 69.6.
  const int64_t tiles_128 = ((M + 127) / 128) * ((N * n_products + 127) / 128);
  if (tiles_128 <= cus / 2 || (small_kernel_takes(Kp, schedule) && tiles_64 <= (Kp >= 768 ? 3 : 2) * (int64_t)cus)) return {0, false};
  // Two workgroups of four waves are resident per compute unit.  The 256 x 128 / 128 x 256 tiles need 6 decode
  // instructions per MFMA, the 128 x 128 tile 8, so the larger tiles win unless they fill the slots much worse.  A last
  // round of at most one workgroup per unit is cheap: alone on its unit a workgroup runs in 0.56 of the time it takes
  // next to another (measured: 252 tiles of 128 x 256 alone, 59 us, against 504 of 128 x 128 in pairs, 55 us).
  const int64_t slots = 2 * (int64_t)cus;
  auto rounds_eff = [&](int bm, int bn) {
    const int64_t tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn) * n_products;
    const int64_t whole = tiles / slots, rest = tiles % slots;
    const double time = (double)whole + (rest == 0 ? 0.0 : (rest <= cus ? 0.564 : 1.0));
    return ((double)tiles / (double)slots) / time;
  };
  struct Cfg { int kernel, bm, bn; double bonus; };
  const Cfg cfgs[3] = {{3, 256, 128, 1.00}, {2, 128, 256, 1.00}, {1, 128, 128, 0.90}};
  int best = 3;
  double best_score = -1.0;
  for (const Cfg& c : cfgs) {
    const double sc = rounds_eff(c.bm, c.bn) * c.bonus;
    if (sc > best_score) {
      best_score = sc;
      best = c.kernel;
    }
  }
  return {best, generated_ok && best >= 2};
}

// Sets of four waves of a workgroup that computes a tile of 128 x 128: two while every tile has a unit to itself, where the
// four waves of one had a SIMD each and waited for every instruction.  us, one set / two: 736 x 4608 x 1536 19.2 / 17.3, 1000 x
// 4096 x 2048 24.7 / 22.3, 800 x 4096 x 4096 41.0 / 36.0, 640 x 6400 x 896 14.6 / 13.8, with gate or residual 2 to 4 more off; x 384
// 9.74 / 9.69.  One order of summation for every shape (LL_GEMM_TILES_COMPILED) needs one set.
constexpr int64_t kTileSetsK = 512;
inline int tile_kernel_sets(int64_t M, int64_t N, int64_t Kp, int n_products, int cus, int schedule) {
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128) * n_products;
  return schedule != 2 /* LL_GEMM_TILES_COMPILED */ && tiles <= cus && Kp >= kTileSetsK ? 2 : 1;
}

// How the small-product kernel divides a launch: 64 x 64 tiles, each by `parts` workgroups that share its K range (steps of
// 256 elements).  Measured when a step took 0.55 us (0.47 now) with one workgroup on every compute unit; handing two to
// four parts over and adding them up takes 2.4 us (their records are read four at a time: five to eight 3.6); with more
// workgroups than units a step takes 0.8 and the launch 2 us more.  us by parts:
//                     tiles, steps    1     2     3     4     5     6     8    12
//   40 x 256 x 5888       4, 23     17.6  13.9  11.8  10.7  11.0  10.9  10.0  10.6
//   48 x 1024 x 4096     16, 16     13.7  12.0  10.8  10.2  11.8  10.3  10.8  11.9
//   64 x 1536 x 6912     24, 27     19.6  15.2  12.9  11.5  12.0  11.7  13.9  16.0
//   130 x 1024 x 4096    48, 16     13.7  12.3  11.1  10.8  11.9  12.7  15.7
//   112 x 2944 x 8192    92, 32     22.8  17.1  17.0  15.3  17.7
//   128 x 3072 x 14336   96, 56     35.9  24.1  24.8  21.8  21.7
//   64 x 3072 x 3072     48, 12     11.5  11.2  10.5  10.1  10.5  12.8  13.3
//   368 x 768 x 3456     72, 14     12.6  11.9  11.1  13.9  14.7  14.3
//   300 x 1024 x 3072    80, 12     11.5  11.5  10.9  12.8  14.3  16.5
//   256 x 3072 x 3072   192, 12     11.9  13.6
// More than four parts gain half a microsecond at most, and below sixteen steps parts gain about one, which is less than what
// they cost a recorded launch (gemm_w4a4_small_kernel<true>).
constexpr int kSmallParts = 4, kSmallPartsSteps = 16;
constexpr int kSmallRecordBytes = 64 * 64 * 4;                            // a part's fp32 sums of its tile
inline int64_t small_product_units(int cus) { return 2 * (int64_t)cus; }  // most (tile, part) pairs of a launch with parts
// Tiles of 64 x 96 where those of 64 x 64 would be more than one per unit and these are not: a step takes 0.71 us against
// 0.9 us for two of the smaller ones (us, 64 x 64 / 64 x 96: 512 x 3072 x 3072 15.2 / 13.7, 736 x 1536 x 1536 9.9 / 9.4, x
// 8960 33.3 / 30.5, 440 x 3072 x 14336 50.4 / 45.2).  Larger ones were measured too: 64 x 128 and 96 x 128 were never ahead
// of both, 128 x 128 by 6 % on 2048 x 2048 x 3072.
// Two sets of four waves (one workgroup per unit, so a second wave on every SIMD) from 2048 elements of K on: a step then takes
// 0.71 us where every unit is busy, with one set 0.83, and the sets' sums meet at the end.  us, one set / two, the product by
// itself: 736 x 1536 x 8960 33.9 / 30.2, 512 x 3072 x 14336 53.2 / 47.0, 736 x 1536 x 2304 12.75 / 12.55, x 2048 11.9 / 11.8, but 512 x
// 3072 x 1792 11.5 / 11.7, 736 x 1536 x 1536 10.4 / 10.5, 512 x 3072 x 1024 9.0 / 9.3; a call of a linear layer, its quantization with
// it: 736 x 1536 x 8960 43.0 / 38.8, x 6144 34.5 / 31.9, x 3072 22.95 / 22.2, x 2560 20.3 / 19.95, x 2304 19.2 / 19.0, x 2048 18.2 / 18.2, 512 x
// 3072 x 14336 59.6 / 54.5, x 4096 24.6 / 23.8, x 2560 19.3 / 19.0, x 2048 18.0 / 18.0, 450 x 2816 x 3328 22.15 / 21.4.  The same on two other
// cards, but 512 x 3072 x 3072 21.1 / 20.4 on one and 21.1 / 21.1 to 21.5 on the others.
constexpr int64_t kSmallSetsK = 2048;
struct SmallGemmPlan {
  int fb;  // tiles of 64 rows by 32 fb columns
  int parts;
  int tiles_m, tiles_n_each;
  int64_t tiles;
  int sets;  // of four waves: K steps are dealt to one or two
};
inline SmallGemmPlan plan_small_gemm(int64_t M, int64_t N, int64_t Kp, int n_products, int cus) {
  SmallGemmPlan p{2, 1, (int)((M + 63) / 64), (int)((N + 63) / 64), 0, 1};
  p.tiles = (int64_t)p.tiles_m * p.tiles_n_each * n_products;
  if (const int64_t each = (N + 95) / 96, wide = p.tiles_m * each * n_products; Kp >= 1024 && p.tiles > cus && wide <= cus) {
    p.fb = 3;
    p.tiles_n_each = (int)each;
    p.tiles = wide;
    p.sets = Kp >= kSmallSetsK ? 2 : 1;
    return p;
  }
  const int64_t steps = (Kp + 255) / 256;
  if (steps < kSmallPartsSteps) return p;
  double best = 0.0;
  for (int64_t s = 1; s <= kSmallParts && (s == 1 || p.tiles * s <= small_product_units(cus)); ++s) {
    const bool beyond = p.tiles * s > cus;
    const double time = (double)((steps + s - 1) / s) * (beyond ? 0.8 : 0.55) + (s > 1 ? 2.4 : 0.0) + (beyond ? 2.0 : 0.0);
    if (s == 1 || time < best) {
      best = time;
      p.parts = (int)s;
    }
  }
  return p;
}

}  // namespace ll
