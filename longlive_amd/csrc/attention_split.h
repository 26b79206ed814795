// How an attention launch is divided between its workgroups: the arithmetic shared by the kernel (device), the
// launcher (host) and the host-side checks of the test suite.  Everything here is integer arithmetic on a few
// launch-wide numbers, identical on both sides.
//
// A launch has tiles (head x group of queries) of n_iter iterations (128 keys each) and G workgroups.  Tiles whose group of
// queries is full come first in the numbering, the heads' last, partly filled groups behind them: the waves of such a tile
// that have no queries skip the matrix work, so an iteration of it costs less (`light` sixteenths of a full one) when the
// busy waves are few enough to have a SIMD each.  Workgroup g first runs `whole_rounds` whole tiles (tile j * G + g in
// round j); workgroups [0, extra) then run one more whole tile each (tile whole_rounds * G + g) and are done.  The tiles
// behind those, numbered from 0 as "split tiles", are cut into units = split tiles x n_iter, and the workgroups [extra, G)
// divide them into shares of equal cost, each cut at tile boundaries into segments and walked from the end backwards.
#pragma once
#include <stdint.h>

#ifndef __HIPCC__
#define LL_SPLIT_FN inline
#else
#define LL_SPLIT_FN __host__ __device__ __forceinline__
#endif

namespace ll {

constexpr uint32_t kFullUnitCost = 16;

struct Division {
  uint32_t G;             // workgroups
  uint32_t whole_rounds;  // whole tiles every workgroup runs first
  uint32_t extra;         // workgroups [0, extra) run one more whole tile and take no share of the split part
  uint32_t n_iter;        // iterations (units) per tile
  uint32_t units;         // units of the split part
  uint32_t full_units;    // of which the first full_units belong to full tiles (cost kFullUnitCost each)
  uint32_t light;         // cost of each unit behind them
};

LL_SPLIT_FN uint64_t cost_before_unit(const Division& d, uint32_t u) {
  return u <= d.full_units ? (uint64_t)kFullUnitCost * u
                           : (uint64_t)kFullUnitCost * d.full_units + (uint64_t)d.light * (u - d.full_units);
}
LL_SPLIT_FN uint64_t split_cost(const Division& d) { return cost_before_unit(d, d.units); }

// First unit of workgroup g's share (g = G: one past the last unit).  Share boundaries sit at equal distances in
// cost and are rounded down to whole units.
LL_SPLIT_FN uint32_t first_unit_of(uint32_t g, const Division& d) {
  if (g <= d.extra) return 0u;
  const uint64_t at = (uint64_t)(g - d.extra) * split_cost(d) / (d.G - d.extra);
  const uint64_t full_cost = (uint64_t)kFullUnitCost * d.full_units;
  return at <= full_cost ? (uint32_t)(at / kFullUnitCost) : d.full_units + (uint32_t)((at - full_cost) / d.light);
}

// The workgroup whose share holds unit u: the g with first_unit_of(g) <= u < first_unit_of(g + 1).
LL_SPLIT_FN uint32_t holder_of_unit(uint32_t u, const Division& d) {
  return d.extra + (uint32_t)((cost_before_unit(d, u + 1) * (d.G - d.extra) - 1) / split_cost(d));
}

struct Segment {
  uint32_t tile;   // tile number in the launch (whole tiles first, split tiles behind them)
  int begin, end;  // iterations [begin, end) of the tile
};

// Position of a workgroup in its work: whole tiles done, and the end of what is left of its share of the units.
struct WorkCursor {
  uint32_t round;
  uint32_t share_end;
};

LL_SPLIT_FN WorkCursor start_of_work(uint32_t g, const Division& d) {
  return WorkCursor{0u, d.units ? first_unit_of(g + 1, d) : 0u};
}

// The next segment of workgroup g, or false when its work is done.
LL_SPLIT_FN bool next_segment(WorkCursor& at, uint32_t g, const Division& d, Segment& seg) {
  if (at.round < d.whole_rounds || (at.round == d.whole_rounds && g < d.extra)) {
    seg.tile = at.round * d.G + g;
    seg.begin = 0;
    seg.end = (int)d.n_iter;
    ++at.round;
    return true;
  }
  if (d.units == 0) return false;
  const uint32_t share_begin = first_unit_of(g, d);
  if (at.share_end <= share_begin) return false;
  const uint32_t split_tile = (at.share_end - 1) / d.n_iter;
  const uint32_t tile_first_unit = split_tile * d.n_iter;
  seg.tile = d.whole_rounds * d.G + d.extra + split_tile;
  seg.begin = share_begin > tile_first_unit ? (int)(share_begin - tile_first_unit) : 0;
  seg.end = (int)(at.share_end - tile_first_unit);
  at.share_end = tile_first_unit + (uint32_t)seg.begin;
  return true;
}

// The workgroups that hold a part of split tile `split_tile`: g_first .. g_last, every one of them (the launcher
// leaves no workgroup of [extra, G) without a unit).
LL_SPLIT_FN void parts_of_tile(uint32_t split_tile, const Division& d, uint32_t& g_first, uint32_t& g_last) {
  g_first = holder_of_unit(split_tile * d.n_iter, d);
  g_last = holder_of_unit(split_tile * d.n_iter + d.n_iter - 1, d);
}

// Which of its two records workgroup g uses for its part of `split_tile`: the first one for the first tile it
// touches, the second one otherwise (only the first and the last tile of a share can be partial).
LL_SPLIT_FN uint32_t record_of_part(uint32_t g, uint32_t split_tile, const Division& d) {
  const uint32_t first_tile = first_unit_of(g, d) / d.n_iter;
  return 2 * g + (first_tile == split_tile ? 0u : 1u);
}

// First iteration of part `part` of a tile of n_iter iterations in `parts` parts (part = parts: one past the last).
LL_SPLIT_FN int first_iteration_of_part(uint32_t part, uint32_t parts, int n_iter) { return (int)(part * (uint32_t)n_iter / parts); }

// ---- short launches (host): waves per workgroup with which kv_attention_short_kernel takes a launch, 0 for the tile
// kernels.  It converts K and V once per 32 queries and fills a compute unit with one workgroup of eight or two of
// four waves, so it is ahead while everything runs at once and the key range is short (us, tile kernels / 8 waves /
// 4 waves; "a + b" = cached + chunk keys in tiles of 32; taken when this kernel rescaled its sums in steps of 2^8, those of
// 2^2 that it has now cost 1 to 2.5 % and move no line by a measured point):
//   G <= CUs      368 queries x 16 heads, 0 + 46 tiles 36.8 / 16.9 / 20.3; 512 x 16, 64 + 16: 36.9 / 28.8 / 31.2;
//                 1024 x 6, 64 + 32: 42.5 / 32.9 / 36.5, but 128 + 32: 48.5 / 50.1 / 57.7 (the divided tiles use all units)
//   up to 12 tiles four waves have two or three tiles each and half the merge: 64 x 12, 0 + 4: 8.4 / 6.7 / 5.8
//   G <= 2 CUs    736 x 12, 0 + 16: 16.3 / 18.4 / 13.7; 512 x 24, 32 + 16: 34.7 / 38.3 / 32.8, but 46 + 23 on 736 x 12:
//                 38.7 / 49.9 / 43.5;   G > 2 CUs: 736 x 24, 0 + 16: 16.8 / 26.4 / 20.5
// A cached tile costs about half as much again as one of the chunk (conversion).  Launches of more than 256 queries per
// head for every head take it over up to 16 tiles (3520 x 2, 0 + 16: 15.4 / 10.4 / 10.5); over more the measurements end at
// one point (700 queries of 2 heads over 900 keys: 12.9 us here, 27.8 in 256-query tiles), and 128-query tiles that share
// their key ranges (plan_narrow_split) have taken most of what there was to gain.
// `policy`: only the automatic choice (-1) and the division without shared tiles (0) take this kernel.  The launch, the
// plan query and the reserve call all ask here.
inline int short_kernel_waves(int64_t Lq, int H, int64_t n_cached, int64_t n_new, int cus, int policy) {
  if (policy > 0) return 0;
  const int64_t groups = H * ((Lq + 31) / 32), cached = (n_cached + 31) / 32, fresh = (n_new + 31) / 32;
  const int64_t length = cached + cached / 2 + fresh;
  if (Lq > 256 * (int64_t)H && length > 16) return 0;
  if (groups <= cus) return length > 176 ? 0 : (cached + fresh <= 12 ? 4 : 8);
  return groups <= 2 * (int64_t)cus && length <= 64 ? 4 : 0;
}

// ---- the launcher's choice (host).  Costs are in iterations of the 128-query kernel; whole rounds of workgroups
// count in full.
struct AttentionPlan {
  int mode;             // LL_ATTENTION_NARROW / WIDE / SPLIT
  int queries;          // per tile: 128 (NARROW, and SPLIT where plan_narrow_split is taken) or 256
  int parts;            // 128-query tiles: workgroups that share the key range of each
  int n_qtiles;         // query tiles per head
  int full_qtiles;      // of which this many come first in the tile numbering (all of them unless mode is SPLIT)
  Division d;           // G = workgroups of the launch; units = 0 unless mode is SPLIT
  int64_t split_tiles;  // tiles of the split part
};

// The cost of a plan for the automatic choice, in the same unit, goes to `cost` (if asked for).
// `allow_split` false leaves the split division out of the automatic choice (a launch that may not use the memory
// partial tiles pass through).
inline AttentionPlan plan_attention(int64_t Lq, int H, int64_t n_keys, int cus, int policy, bool allow_split = true,
                                    double* cost = nullptr) {
  constexpr double kWideIteration = 1.64;  // an iteration of the 256-query kernel takes this much longer for twice the work
  constexpr double kCombine = 6.0;         // partial results when every workgroup shares: writing, counting, combining
  constexpr double kCombineFew = 1.5;      // the same when only the workgroups without a whole extra tile share
  constexpr double kRound = 4.0;           // what a workgroup spends per tile outside the iterations (Q, first K/V
                                           // tile, output); fitted on 256 .. 2640 keys, where it decides
  const int64_t n_iter = (n_keys + 127) / 128;
  const int64_t tiles_narrow = H * ((Lq + 127) / 128);
  const int64_t nq = (Lq + 255) / 256;
  const int64_t tiles_wide = H * nq;
  // The last group of queries of every head holds `rest` of 256 queries.  With at most 128 of them every wave
  // that has queries has its SIMD to itself (waves w and w + 4 share one) and the tile is light: the other waves
  // only help to bring K and V in (measured: 0.68 of the time of a full tile with three of eight waves busy, and
  // 12 sixteenths weighing better than 11 with four).
  // With more, some SIMD carries two busy waves as in a full tile, and the tile counts as full.
  const int64_t rest = Lq - (nq - 1) * 256;
  const int64_t light_tiles = rest <= 128 ? H : 0, full_tiles = tiles_wide - light_tiles;
  const uint32_t light = (uint32_t)(8 + (rest + 31) / 32);  // 9 .. 12 for one to four busy waves

  // Split: `rounds` whole rounds of full tiles, `extra` more whole full tiles on the first workgroups, the rest of
  // the tiles in shares of equal cost for the other workgroups.  Two shapes are weighed against each other:
  //  (a) every left-over full tile runs whole and only the light tiles are shared out, among the workgroups that
  //      have no left-over tile - no tile is combined that need not be;
  //  (b) no extra tiles, all workgroups share everything behind the whole rounds.  A handful of left-over tiles
  //      would be cut into many thin parts each (and combined by a single workgroup): then one whole round joins
  //      the split part, whose shares are a little more than one tile.
  struct Shape { int64_t rounds, extra; double cost; };
  auto weigh = [&](int64_t rounds, int64_t extra) {
    Shape sh{rounds, extra, 1e300};
    const int64_t split_full = full_tiles - rounds * cus - extra, servers = cus - extra;
    if (rounds < 0 || extra < 0 || split_full < 0 || servers < 1) return sh;
    const int64_t cost = n_iter * ((int64_t)kFullUnitCost * split_full + (int64_t)light * light_tiles);
    if (cost == 0) return sh;  // nothing to split
    // every sharing workgroup needs a unit when others run whole tiles too (the parts of a tile are counted by shares)
    if ((rounds > 0 || extra > 0) && cost < (int64_t)kFullUnitCost * servers) return sh;
    const double share = (double)((cost + servers - 1) / servers) / kFullUnitCost;
    sh.cost = kWideIteration * ((double)(rounds * n_iter) + (extra > 0 && share < (double)n_iter ? (double)n_iter : share)) +
              kRound * (double)(rounds + 1) + (extra > 0 ? kCombineFew : kCombine);
    return sh;
  };
  int64_t rounds_b = full_tiles / cus;
  if (const int64_t left = tiles_wide - rounds_b * cus; left > 0 && left * 4 < cus && rounds_b > 0) --rounds_b;
  Shape best = weigh(rounds_b, 0);
  if (light_tiles > 0 && full_tiles % cus > 0) {
    // (a) is taken unless (b) promises more than 4 %: where the two are that close (configs[2]: 107 against 104
    // iterations) they measure the same to half a per cent, and (a) combines 8 tiles instead of 263.
    const Shape a = weigh(full_tiles / cus, full_tiles % cus);
    if (a.cost <= best.cost * 1.04) best = a;
  }
  if (!allow_split) best.cost = 1e300;
  const double cost_narrow = (double)((tiles_narrow + cus - 1) / cus) * ((double)n_iter + kRound);
  const double cost_wide = (double)((tiles_wide + cus - 1) / cus) * (kWideIteration * (double)n_iter + kRound);
  int mode = cost_narrow <= cost_wide && cost_narrow <= best.cost ? 0 : (cost_wide <= best.cost ? 1 : 2);
  if (cost) *cost = mode == 0 ? cost_narrow : mode == 1 ? cost_wide : best.cost;
  if (policy >= 0) mode = policy;
  if (tiles_wide * n_iter >= (1ll << 31)) mode = 0;  // units are counted in 32 bits (costs in 64)
  if (mode == 2 && best.cost >= 1e300) mode = 1;     // nothing that could be split
  AttentionPlan plan{};
  plan.mode = mode;
  plan.d.whole_rounds = 1;
  plan.d.n_iter = (uint32_t)n_iter;
  plan.d.light = kFullUnitCost;
  plan.queries = mode == 0 ? 128 : 256;
  plan.parts = 1;
  if (mode == 0) {
    plan.n_qtiles = plan.full_qtiles = (int)((Lq + 127) / 128);
    plan.d.G = (uint32_t)tiles_narrow;
  } else {
    plan.n_qtiles = plan.full_qtiles = (int)nq;
    plan.d.G = (uint32_t)tiles_wide;
    if (mode == 2) {
      const int64_t split_full = full_tiles - best.rounds * cus - best.extra;
      plan.full_qtiles = (int)(light_tiles ? nq - 1 : nq);
      plan.d.whole_rounds = (uint32_t)best.rounds;
      plan.d.extra = (uint32_t)best.extra;
      plan.split_tiles = split_full + light_tiles;
      plan.d.units = (uint32_t)(plan.split_tiles * n_iter);
      plan.d.full_units = (uint32_t)(split_full * n_iter);
      plan.d.light = light_tiles ? light : kFullUnitCost;
      // without whole tiles no workgroup may be left without a unit either
      const uint64_t cost = split_cost(plan.d);
      const uint64_t shares = cost < kFullUnitCost ? 1 : cost / kFullUnitCost;  // a single light unit costs less than 16
      plan.d.G = (uint32_t)(best.rounds == 0 && best.extra == 0 && shares < (uint64_t)cus ? shares : (uint64_t)cus);
    }
  }
  return plan;
}

// The memory of a split division.  A workgroup's partial result: per wave 64 (256-query tiles) or 32 (128) O^T registers, reference
// point and row sum, per lane; a share of 256-query tiles may end one tile and begin another.
constexpr size_t partial_bytes(int queries) { return (size_t)8 * (queries / 4 + 2) * 64 * sizeof(float); }
inline size_t partial_records(const AttentionPlan& plan) { return (plan.queries == 128 ? 1 : 2) * (size_t)plan.d.G; }

// Split division with tiles of 128 queries: the key range of every tile shared by the same number of workgroups (`parts`), all
// in one round, each with one run of iterations.  Returns its cost in iterations of the 128-query kernel, 2 us each.  us, by
// parts (in brackets: whole 128-query tiles / shares of 256-query tiles, which cross tiles and then pay for two prologues,
// two exchanges and the 64-bit arithmetic of the shares):
//    736 queries x 12, 1472 cached + 736 keys   31.6 (2) 27.4 (3)                   [44.3 / 40.4]
//   1408 x 4, 2816 + 1408                       46.1 (2) 37.7 (3) 31.3 (4) 31.5 (5) [75.3 / 46.8]
//   1760 x 8, 3520 + 1760                       58.2 (2)                            [91.8 / 63.2]
//   2000 x 6, 0 + 2000                          29.7 (2)                            [39.4 / 38.7]
//   3520 x 2, 7040 + 3520                       96.1 (2) 70.4 (3) 58.2 (4)          [172 / 70.3]
//    512 x 4, 1024 + 512                        24.5 (2) 21.1 (3) 19.3 (4) 20.9 (5) 19.6 (6) 19.5 (8) 22.1 (12)
//    736 x 12, 0 + 512                          17.6 (2) 18.0 (3)                   [15.6 / 25.1]
// Two rounds of parts (880 x 24, 0.88 k + 880: 47.5 with three parts) lose against whole tiles (38.2).
// Iterations take longer as the last tenth of the compute units joins in, which decides over long ranges; there shares of
// 256-query tiles are ahead, most of all where four of them make up a tile and none crosses to the next (us, two parts /
// shares): 2624 x 6 over 10496 107.4 / 103.1, 3200 x 5 over 9600 99.4 / 96.7, 1936 x 8 over 7744 84.1 / 80.8, 2000 x 8 over
// 8946 90.8 / 88.8, but 2624 x 6 over 6471 71.6 / 73.1, 1000 x 16 over 5000 58.8 / 60.4.
inline double plan_narrow_split(int64_t Lq, int H, int64_t n_keys, int cus, AttentionPlan& plan) {
  constexpr double kRound = 4.0, kExchange = 2.5, kPerPart = 0.5, kFullChip = 0.8, kSpared = 1.0;
  const int64_t n_iter = (n_keys + 127) / 128, nq = (Lq + 127) / 128, tiles = H * nq;
  int64_t parts = 0;
  double best = 1e300;
  for (int64_t s = 2; s * tiles <= cus && s <= n_iter; ++s) {
    const double cost = (double)((n_iter + s - 1) / s) + kRound + kExchange + kPerPart * (double)s;
    if (cost < best) {
      best = cost;
      parts = s;
    }
  }
  if (parts < 2) return 1e300;
  plan = AttentionPlan{};
  plan.mode = 2;
  plan.queries = 128;
  plan.parts = (int)parts;
  plan.n_qtiles = plan.full_qtiles = (int)nq;
  plan.d.G = (uint32_t)(tiles * parts);
  plan.d.n_iter = (uint32_t)n_iter;
  plan.split_tiles = tiles;
  const double longer = kFullChip * ((double)(tiles * parts) / cus - 0.9) * (double)((n_iter + parts - 1) / parts);
  return best + (longer > kSpared ? longer - kSpared : 0.0);
}

// The division of a launch that the short kernel does not take, under `policy`.  The split division has tiles of 128 queries
// where these are the cheapest division of all under the automatic choice.
inline AttentionPlan plan_division(int64_t Lq, int H, int64_t n_cached, int64_t n_new, int cus, int policy, bool allow_split = true) {
  // What shares of 256-query tiles cost beyond plan_attention's estimate: where they cross tiles (40 instead of 30 us on the
  // first shape above), and where up to four of them make up each tile.
  constexpr double kCrossing = 5.0, kWhole = 4.5;
  double cost = 0.0;
  const AttentionPlan plan = plan_attention(Lq, H, n_cached + n_new, cus, policy == 2 ? -1 : policy, allow_split, &cost);
  const bool may_split = policy == 2 /* LL_ATTENTION_SPLIT */ || (policy == -1 /* LL_ATTENTION_AUTO */ && allow_split);
  if (may_split && !short_kernel_waves(Lq, H, n_cached, n_new, cus, -1)) {
    AttentionPlan narrow;
    const bool whole = plan.mode == 2 && plan.d.whole_rounds == 0 && plan.d.extra == 0 && plan.d.full_units == plan.d.units &&
                       plan.d.G % plan.split_tiles == 0 && plan.d.G <= 4 * plan.split_tiles;
    if (plan_narrow_split(Lq, H, n_cached + n_new, cus, narrow) < cost + (plan.mode != 2 ? 0.0 : whole ? kWhole : kCrossing)) return narrow;
  }
  return policy == 2 ? plan_attention(Lq, H, n_cached + n_new, cus, policy, allow_split) : plan;
}

}  // namespace ll
