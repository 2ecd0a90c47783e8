// How a prefill call is cut into workgroups: the key groups that the waves of
// a workgroup form (gqa_prefill_kernel), and the number of workgroups that a
// row's key range is split over. Host code without HIP.
#pragma once

#include <algorithm>
#include <cstdint>

namespace sai {

// Key groups the kernel can form: as many as tiles fit the LDS at once. Above
// head_dim 128 one: two int8 tiles fit, but their loads do not fit the
// registers beside the query (56 to 103 spilled).
constexpr int prefill_max_key_groups(int head_dim, bool int4) {
  return head_dim > 128 ? 1 : (int4 ? 2 : 4);
}

// Row blocks of 16 attention rows per wave, and rows (query positions x heads
// of one kv head) of a workgroup of eight waves.
constexpr int prefill_row_blocks(int head_dim, int key_groups) {
  return head_dim > 128 || key_groups == 4 ? 1 : 2;
}
constexpr int prefill_workgroup_rows(int head_dim, int key_groups) {
  return 16 * prefill_row_blocks(head_dim, key_groups) * (8 / key_groups);
}

struct PrefillShape {
  int head_dim;  // stored width
  bool int4;
  int group, kv_heads, batch;
  int sq;        // new tokens per sequence
  int64_t past;  // the longest sequence's cached tokens
  int window;    // visible keys per query (0: all)
  int cus;
};

struct PrefillPlan {
  int key_groups = 1;
  int key_splits = 1;
  int split_tiles = 0;  // 64-token tiles of a split (key_splits > 1)
};

// 64-token tiles that the rows of new positions [q0, q1) read, at most,
// whatever the sequence's length up to `past`: W + q1 - q0 - 1 neighbouring
// keys with a window.
inline int64_t prefill_tiles(const PrefillShape& s, int q0, int q1) {
  const int64_t all = (s.past + q1 - 1) / 64 + 1;
  if (s.window <= 0) return all;
  return std::min(all, ((int64_t)s.window + (q1 - q0) + 61) / 64 + 1);
}

// Microseconds of a call whose workgroups run at once: fixed (launches, query,
// first loads, output), for each tile of the longest workgroup, and on top for
// each of its tiles that needs the causal mask. Fitted to 2000 timings of 840
// shapes, all splits and key groups that fit (median error 4 %).
struct PrefillCost {
  float fixed, tile, edge;
};
inline PrefillCost prefill_cost(int head_dim, bool int4, int key_groups) {
  const bool d64 = head_dim <= 64;
  if (int4) {
    if (head_dim > 128) return {8.0f, 4.47f, 0.8f};
    if (key_groups == 1) return d64 ? PrefillCost{7.8f, 2.07f, 0.8f} : PrefillCost{10.4f, 3.24f, 0.8f};
    return d64 ? PrefillCost{8.0f, 1.56f, 1.1f} : PrefillCost{11.3f, 2.11f, 1.1f};
  }
  if (head_dim > 192) return {8.3f, 3.03f, 1.4f};
  if (head_dim > 128) return {6.9f, 2.65f, 1.4f};
  if (key_groups == 1) return d64 ? PrefillCost{7.7f, 1.63f, 1.8f} : PrefillCost{10.0f, 2.39f, 1.8f};
  if (key_groups == 2) return d64 ? PrefillCost{7.8f, 1.18f, 1.0f} : PrefillCost{12.2f, 1.43f, 1.0f};
  return d64 ? PrefillCost{6.9f, 0.74f, 0.4f} : PrefillCost{8.2f, 0.91f, 0.4f};
}

// The cheapest of the splits that a call can take, by the costs above. Two key
// groups pass a tile in 0.6 (head_dim 64: 0.72) of the time, but take twice the
// workgroups for the same rows, which pays only while these still fit the CUs
// (one each) or are mostly empty anyway; a split of the key range fills idle
// CUs, but every row's partials are written and read again by another launch.
// No threshold on the number of workgroups gets both right. us per call at
// 32Q/8KV, int8 (key groups x splits):
//                               1x1    1x2    1x4    2x1    2x2
//   128:  6 x 256 over 4000     178    210           221
//         1 x 1200               58     68            55
//         1 x 1000               50     48            36
//         1 x 600 over 4000     189           124    118    134
//         1 x 400 over 4000     179                  114     75
//    64:  1 x 1000 over 4000    148     92           110    124
// Four groups (int8; 32 rows a workgroup) serve every chunk of at most 32 rows
// a kv head (16 x 8 over 4000: 86 / 70 / 52 us with 1 / 2 / 4). A split keeps
// at least two rounds of tiles; ranges below 16 tiles are not split.
inline PrefillPlan prefill_plan(const PrefillShape& s) {
  const int64_t rows = (int64_t)s.sq * s.group;
  const int max_groups = prefill_max_key_groups(s.head_dim, s.int4);
  PrefillPlan best;
  double best_us = -1.0;
  bool few = true;  // 256-row workgroups do not fill the CUs
  for (int kg = 1; kg <= max_groups; kg *= 2) {
    const int qt = prefill_workgroup_rows(s.head_dim, kg) / s.group;
    const int blocks = (s.sq + qt - 1) / qt;
    const int64_t wgs = (int64_t)blocks * s.kv_heads * s.batch;
    if (kg == 1) few = wgs < s.cus;
    if (max_groups == 4 && (rows <= 32) != (kg == 4)) continue;
    if (!few && rows > 128) break;  // one key group, no split
    int64_t tiles = 0, least = INT64_MAX, edge = 0;
    for (int i = 0; i < blocks; ++i) {
      const int q0 = i * qt, q1 = std::min(s.sq, q0 + qt);
      const int64_t n = prefill_tiles(s, q0, q1);
      tiles = std::max(tiles, n);
      least = std::min(least, n);
      edge = std::max(edge, (s.past + q1 - 1) / 64 + 1 - (s.past + q0 + 1) / 64);
    }
    // with equal work a second round of workgroups starts when the first ends;
    // causal rows of different lengths fill it
    const double even = (double)least / (double)tiles, fill = (double)wgs / s.cus;
    const double rounds =
        fill <= 1.0 ? 1.0 : (1.0 - even) * fill + even * (double)((wgs + s.cus - 1) / s.cus);
    const PrefillCost c = prefill_cost(s.head_dim, s.int4, kg);
    const int64_t max_splits =
        tiles < 16 ? 1 : std::max<int64_t>(1, std::min(s.cus / wgs, tiles / std::max(4, 2 * kg)));
    for (int64_t n = 1; n <= max_splits; ++n) {
      const int64_t per = (tiles + n - 1) / n;
      const int64_t steps = (per + kg - 1) / kg * kg;  // a group's tiles, times kg
      const int64_t edges = (std::min(edge, per) + kg - 1) / kg;
      double us = rounds * (c.fixed + c.tile * (double)steps + c.edge * (double)edges);
      // the merge: its launch, and the partials' bytes
      if (n > 1)
        us += 0.7 + (double)(rows * s.kv_heads * s.batch * n * (s.head_dim + 2)) * 8.0 / 3.6e6;
      if (best_us >= 0.0 && us >= best_us) continue;
      best_us = us;
      best.key_groups = kg;
      best.split_tiles = (int)per;
      best.key_splits = (int)((tiles + per - 1) / per);
    }
  }
  return best;
}

}  // namespace sai
