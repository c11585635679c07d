// Which tile of tiled_gemm.h an unsplit product takes: a time model per tile
// shape, fitted to measurements, and the shape (or pair of shapes on two
// column ranges) it predicts fastest.  Host code, shared by the launchers.
#pragma once

#include <stdint.h>

namespace mi355 {
namespace tiled {

// Predicted us of a [rows, k] x [cols, k] product on bm x bn tiles:
//   c0 + round * rounds
//      + (K steps of 64) * (full rounds * step[occ - 1] + last round's step
//                           + load * tiles per CU)
//      + weight * (MB of weights)
// where a round is occ workgroups on every CU, and a last round that needs
// only w of them per CU costs step[w - 1].  step[w - 1] is the part of a K
// step that a CU with w workgroups waits for whether or not the others work;
// `load` the part that follows the work of the whole chip (a fully loaded
// chip lowers its clock: 1.8 GHz under these kernels at long prompts).  The
// constants are least-squares fits (non-negative) to sweeps on MI355X over the
// Qwen2.5-0.5B to 14B projections at 33 - 4096 rows, weights rotated through
// HBM, made before the epilogue stored whole row segments and loaded its scales
// together.  Against the kernels as they are the chosen launches' mean error is
// 7% for the 16-bit linear and both gate/ups and 13% for the int8 linear, which
// is predicted 12% high throughout (bench.py --only tile-plans).
// `round` is a tile's first loads and its epilogue, which nothing overlaps
// where a CU holds one workgroup.
struct ShapeCost {
  int bm, bn, threads, occ;  // threads per workgroup
  double c0, step[3], load, weight, round;
  double least;  // a K step of a last round takes no less, however few its tiles
};

// (32-bit divisions: the plan runs in every call; with 64-bit ones it cost a
// call about 0.6 us, as here, with constant tile sizes, 0.02 us.)
inline uint32_t plan_cdiv(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// The time of a launch that holds 2^32 threads or more, which the runtime
// refuses: 65 - 512 rows of 2^28 columns and more reach that with small tiles,
// where larger ones (fewer threads per output element) still hold them.
constexpr double kNoLaunch = 1e30;

__attribute__((always_inline)) inline double shape_time(const ShapeCost& s, uint32_t rows, uint32_t cols, uint32_t k,
                                                        double wmb, uint32_t cus) {
  const uint64_t all = static_cast<uint64_t>(plan_cdiv(rows, static_cast<uint32_t>(s.bm))) *
                       plan_cdiv(cols, static_cast<uint32_t>(s.bn));
  if (all > 0xffffffffu / static_cast<uint32_t>(s.threads)) return kNoLaunch;
  const uint32_t tiles = static_cast<uint32_t>(all);
  const uint32_t slots = cus * static_cast<uint32_t>(s.occ);
  const uint32_t full = tiles / slots, rest = tiles - full * slots;
  double per_step = full * s.step[s.occ - 1] + s.load * tiles / cus;
  if (rest > 0) {
    const double last = s.step[(rest > cus) + (rest > 2 * cus)];
    per_step += last;
    if (s.least > 0) {
      const double with_load = last + s.load * rest / cus;
      if (with_load < s.least) per_step += s.least - with_load;
    }
  }
  return s.c0 + s.round * (full + (rest > 0)) + plan_cdiv(k, 64u) * per_step + s.weight * wmb;
}

struct TilePlan {
  int shape;        // the one shape, or the leading columns'
  int lead;         // leading columns of a two-launch plan (0: one launch)
  int tail;         // the remaining columns' shape (lead > 0)
  double cost;      // predicted us
};

// The fastest single shape of the table; with `split`, also every pair of
// launches that gives the leading columns whole rounds of one shape and the
// remaining columns another, so a last, thinly filled round of large tiles
// becomes a round of small ones.  (A round need not end at a column boundary:
// the lead's tiles fill its rounds in order.)  wmb: MB of weights over all n
// columns.
template <int N>
__attribute__((always_inline)) inline TilePlan plan_tiles(const ShapeCost (&table)[N], uint32_t rows, uint32_t n,
                                                          uint32_t k, double wmb, uint32_t cus, bool split) {
  TilePlan best{0, 0, 0, kNoLaunch};
#pragma unroll
  for (int i = 0; i < N; ++i) {  // unrolled: the table's tile sizes become constants
    const double c = shape_time(table[i], rows, n, k, wmb, cus);
    if (c < best.cost) best = TilePlan{i, 0, 0, c};
  }
  if (!split) return best;
  constexpr double kSecondLaunch = 1.7;  // us, of the same fits
  for (int i = 0; i < N; ++i) {
    const ShapeCost& s = table[i];
    const uint32_t tiles_m = plan_cdiv(rows, static_cast<uint32_t>(s.bm));
    const uint32_t slots = cus * static_cast<uint32_t>(s.occ);
    const uint32_t full = plan_cdiv(n, static_cast<uint32_t>(s.bn)) * tiles_m / slots;
    if (full < 1) continue;
    const uint32_t lead = full * slots / tiles_m * static_cast<uint32_t>(s.bn);
    if (lead == 0 || lead >= n) continue;
    const double share = static_cast<double>(lead) / n;
    const double head = shape_time(s, rows, lead, k, wmb * share, cus) + kSecondLaunch;
    if (head >= best.cost) continue;
    for (int j = 0; j < N; ++j) {
      const double c = head + shape_time(table[j], rows, n - lead, k, wmb * (1 - share), cus);
      if (c < best.cost) best = TilePlan{i, static_cast<int>(lead), j, c};
    }
  }
  return best;
}

// Small tiles for 17 - 64 rows of the two linears: 32 x 64 or, for n > 10000,
// 32 x 128 up to 32 rows, 64 x 64 above.  They read each weight byte once and x
// once per workgroup, where skinny tiles re-load x for every weight piece or
// the weights per 32-row tile, but only win with >= 128 tile columns to spread
// over the CUs (a sweep over the Qwen2.5-1.5B / 7B projections at 16 - 64 rows:
// int8 gate/up 7B, 32 rows 85.1 -> 40.7 us, 1.5B 21.3 -> 14.8 us; the 1536-wide
// down and q/o projections 1.8x slower, so they keep weight streaming).
inline uint32_t small_tile_columns(uint32_t rows, uint32_t n) { return rows <= 32 && n > 10000 ? 128u : 64u; }
inline bool small_tiles_pay(uint32_t rows, uint32_t n) {
  return rows > 16 && rows <= 64 && plan_cdiv(n, small_tile_columns(rows, n)) >= 128;
}

// One int8 matrix (w8a16.hip): 64 x 64, 64 x 128, 128 x 128, 192 x 128 (capped
// at 128 registers, two per CU) and 32 x 64.
constexpr ShapeCost kW8Cost[] = {{64, 64, 256, 3, 6.1, {0.181, 0.262, 0.400}, 0.060, 0.050, 0},
                                 {64, 128, 512, 2, 2.8, {0.250, 0.432, 0}, 0.101, 0.026, 3.4},
                                 {128, 128, 512, 2, 3.2, {0.288, 0.557, 0}, 0.216, 0.001, 5.0},
                                 {192, 128, 512, 2, 3.0, {0.429, 0.761, 0}, 0.322, 0, 6.5},
                                 {32, 64, 128, 3, 5.5, {0.177, 0.262, 0.282}, 0.022, 0.052, 0}};
// One 16-bit matrix (linear16.hip): 64 x 64, 128 x 64, 64 x 128, 128 x 128 (one
// and two per CU), 256 x 128 and 256 x 256.  (A step of one 256 x 256 tile is
// 0.86 us of MFMA at the peak rate; the fit had no round of few such tiles and
// priced one of 24 at 0.51 us: 14B down, 3500 rows, 280 tiles, 496 us predicted,
// 613 measured, where 256 x 128 tiles take 534.)
constexpr ShapeCost kL16Cost[] = {{64, 64, 256, 2, 2.0, {0.213, 0.368, 0}, 0, 0.138, 0.8},
                                  {128, 64, 256, 2, 3.2, {0.259, 0.533, 0}, 0.017, 0.126, 1.8},
                                  {64, 128, 512, 1, 1.2, {0.235, 0, 0}, 0.048, 0.164, 2.2},
                                  {128, 128, 512, 1, 1.5, {0.298, 0, 0}, 0.170, 0.126, 3.0},
                                  {128, 128, 512, 2, 2.4, {0.363, 0.433, 0}, 0.263, 0.085, 2.7},
                                  {256, 128, 512, 1, 0, {0.523, 0, 0}, 0.277, 0.011, 9.6},
                                  {256, 256, 512, 1, 0, {0.397, 0, 0}, 1.198, 0, 20.9, 1.05}};
// 16-bit gate/up + SiLU-and-mul (gate_up_silu.hip): 64 x 64, 128 x 64, 128 x
// 128, 192 x 128, 256 x 128 and 256 x 64.
constexpr ShapeCost kGateUpCost[] = {{64, 64, 256, 2, 1.7, {0.328, 0.551, 0}, 0.055, 0.101, 0},
                                     {128, 64, 256, 2, 3.6, {0.347, 0.715, 0}, 0.130, 0.038, 1.5},
                                     {128, 128, 512, 1, 1.6, {0.655, 0, 0}, 0.277, 0.035, 2.7},
                                     {192, 128, 512, 1, 1.3, {0.772, 0, 0}, 0.405, 0.007, 6.6},
                                     {256, 128, 512, 1, 1.4, {0.889, 0, 0}, 0.650, 0, 8.6},
                                     {256, 64, 512, 1, 0.1, {0.516, 0, 0}, 0.261, 0.068, 5.2}};
// Int8 gate/up + SiLU-and-mul (w8a16.hip): 96 x 128, 64 x 64, 128 x 64 (three
// and two per CU), 192 x 128, 256 x 128 and 128 x 64 in the step pipeline.
constexpr ShapeCost kGateUp8Cost[] = {{96, 128, 256, 1, 2.8, {0.639, 0, 0}, 0.113, 0, 6.5},
                                      {64, 64, 256, 3, 5.6, {0.250, 0.446, 0.644}, 0.092, 0.034, 2.7},
                                      {128, 64, 256, 3, 4.4, {0.405, 0.570, 0.917}, 0.167, 0.025, 4.3},
                                      {128, 64, 256, 2, 4.6, {0.382, 0.616, 0}, 0.179, 0.011, 5.4},
                                      {192, 128, 512, 2, 0, {0.914, 2.080, 0}, 0.317, 0, 9.8},
                                      {256, 128, 512, 1, 0, {0.888, 0, 0}, 0.747, 0, 10.5},
                                      {128, 64, 256, 1, 0, {0.620, 0, 0}, 0.030, 0, 5.0}};

}  // namespace tiled
}  // namespace mi355
