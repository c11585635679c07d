// Split-K GEMM for gfx950: the LDS-tiled kernel of tiled_gemm.h over S ranges
// of K (EPI_PART, fp32 sums to a workspace), then one pass that adds the S
// sums of each output in range order and applies the caller's epilogue; plus
// the plan that picks tile and S, for the W8A16 linear (w8a16.hip) and the
// 16-bit linear (linear16.hip).
//
// Why.  Up to a few hundred rows the output of a down projection (n 896 -
// 5120) holds 12 - 100 tiles, and the weights (k 4864 - 18944) are a deep
// stream each tile reads alone: 256 CUs sit mostly idle behind a serial chain
// of 76 - 296 K steps.  S = CUs / tiles ranges give every CU a workgroup and
// cut the chain by S, for 8 S rows n bytes of extra traffic (fp32 sums
// written once and read once, L2 and Infinity Cache hits) and a second
// launch.  Measured on MI355X, fp16, weights from HBM, unsplit (the stream
// kernel or skinny tiles up to 64 rows, the tiles of tiled_plan.h beyond) and
// split, both passes:
//   7B down (18944 -> 3584), 16-bit:  64 rows 79.1 -> 36.9 us, 200 rows 78.4
//     -> 52.6, 512 rows 119 -> 85.5, 1000 rows 167 -> 144;
//     int8: 64 rows 80.5 -> 27.0, 200 rows 76.8 -> 46.0, 512 rows 107 -> 89
//   1.5B down (8960 -> 1536), 16-bit: 64 rows 22.5 -> 13.1, 200 rows 36.1 ->
//     19.4, 512 rows 39.4 -> 29.2; int8: 64 rows 28.7 -> 13.0, 200 rows 34.8
//     -> 19.3, 1000 rows 48.6 -> 43.3
// What bounds it: HBM on the weights up to about 64 rows, per-step latency of one workgroup per CU above;
// the second pass costs about 3 us and its launch about 3 more in a stream.
//
// Every output's sum is taken in one fixed order (range by range, each in
// tiled_gemm's order), so equal calls give equal bits.
#pragma once

#include "common.h"
#include "tiled_gemm.h"
#include "tiled_plan.h"

namespace mi355 {
namespace tiled {

// EPI: the caller's unsplit epilogue (EPI_W8 or EPI_LINEAR); VEC: columns per
// thread (4 with 16-byte loads, or 1).  Bound by latency: a thread's loads of
// 4 ranges are in flight together.
template <typename TO, int EPI, int VEC>
__global__ __launch_bounds__(256) void split_k_reduce(const Params p) {
  static_assert(EPI == EPI_W8 || EPI == EPI_LINEAR, "one matrix");
  const int nv = p.n / VEC;
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (id >= static_cast<int64_t>(nv) * p.rows) return;
  const int64_t m = id / nv;
  const int n = static_cast<int>(id - m * nv) * VEC;
  const int64_t plane = static_cast<int64_t>(p.rows) * p.n;
  const float* src = p.part + m * p.n + n;
  float acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
#pragma unroll 4
  for (int s = 0; s < p.splits; ++s) {
    if constexpr (VEC == 4) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(src + s * plane);
      acc[0] += v.x; acc[1] += v.y; acc[2] += v.z; acc[3] += v.w;
    } else {
      acc[0] += src[s * plane];
    }
  }
  float v[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    if constexpr (EPI == EPI_W8) {
      const float sc = load_dyn(p.scale, n + e, p.sdt);
      v[e] = p.bdt >= 0 ? __builtin_fmaf(acc[e], sc, load_dyn(p.bias, n + e, p.bdt)) : acc[e] * sc;
    } else {
      v[e] = p.bdt >= 0 ? acc[e] + load_dyn(p.bias, n + e, p.bdt) : acc[e];
    }
  }
  const int64_t o = m * p.os + n;
  if constexpr (VEC == 4) {
    if constexpr (is_half_width<TO>::value) {
      const f32x2 lo = {v[0], v[1]}, hi = {v[2], v[3]};
      *reinterpret_cast<u32x2*>(static_cast<typename TO::bits*>(p.out) + o) = u32x2{narrow2<TO>(lo), narrow2<TO>(hi)};
    } else {
      *reinterpret_cast<u32x4*>(static_cast<float*>(p.out) + o) =
          u32x4{as_u32(v[0]), as_u32(v[1]), as_u32(v[2]), as_u32(v[3])};
    }
  } else {
    store_elem<TO>(p.out, o, v[0]);
  }
}

// ---------------------------------------------------------------- the plan

// Time of one call in us over a tile shape: c0 + step * (K steps a CU runs
// one after another) + part * (MB of fp32 sums written and read) + weight *
// (MB of weights).  Least-squares fits of a sweep on MI355X over the
// Qwen2.5-0.5B to 14B down projections and square projections (896 - 5120
// outputs, k 1536 - 18944) at 24 - 1500 rows, weights rotated through HBM: on
// the kernels as they are, mean error 5% (int8 3% high) over the launches it
// chooses at 72 - 4096 rows.
struct TileCost {
  int bm, bn;
  double c0, step, part, weight;
};
enum { SPLIT_TILES = 5 };
// Split tiles: 32 x 128, 64 x 64, 64 x 128, 128 x 128, 256 x 256.
constexpr TileCost kSplitCost16[SPLIT_TILES] = {
    {32, 128, 5.4, 0.256, 0.199, 0.113}, {64, 64, 5.0, 0.202, 0.288, 0.091},  {64, 128, 5.3, 0.310, 0.307, 0.087},
    {128, 128, 6.8, 0.440, 0.230, 0.060}, {256, 256, 2.8, 1.406, 0.219, 0.054}};
constexpr TileCost kSplitCost8[SPLIT_TILES] = {
    {32, 128, 6.4, 0.235, 0.249, 0.082}, {64, 64, 6.3, 0.226, 0.281, 0.053},  {64, 128, 6.8, 0.284, 0.320, 0.054},
    {128, 128, 8.9, 0.430, 0.226, 0.011}, {256, 256, 4.1, 1.659, 0.211, 0.005}};
// The weight-streaming kernel at 17 - 24, 25 - 32, 33 - 48 and 49 - 64 rows
// (from 49 rows of more than 8 MB of int8 weights: the kernels that run
// there): fixed us, us per MB of weights.
constexpr double kStreamCost16[4][2] = {{3.1, 0.24}, {3.4, 0.29}, {4.1, 0.44}, {4.9, 0.52}};
constexpr double kStreamCost8[4][2] = {{3.5, 0.36}, {4.1, 0.44}, {4.5, 0.69}, {4.9, 0.90}};
// The kernels of 17 - 64 rows on outputs of more than kWide columns, which
// those lines do not describe: the stream kernel at 17 - 24 and 25 - 32 rows,
// then 32 x 64, 32 x 128 and 64 x 64 tiles (small_tiles_pay): fixed us, us per
// K step of one and of more workgroups per CU, us per MB of weights and per MB
// and row.  Fits of a sweep on MI355X over 36 outputs of 8192 - 32768 columns
// (k 896 - 18944) at 17 - 64 rows, weights rotated through HBM: mean error 1 -
// 6% per kernel.
struct WideCost {
  double c0, step1, step2, weight, row;
};
constexpr uint32_t kWide = 127 * 64;
constexpr WideCost kWideCost16[5] = {{3.7, 0, 0, 0.152, 0.0025}, {4.8, 0, 0, 0.161, 0.0023},
                                     {4.1, 0.246, 0.246, 0.016, 0.0006}, {0, 0.246, 0.246, 0.115, 0.0005},
                                     {3.5, 0.217, 0.405, 0.051, 0.0007}};
constexpr WideCost kWideCost8[5] = {{6.2, 0, 0, 0.171, 0.0043}, {7.9, 0, 0, 0.199, 0.0039},
                                    {4.3, 0.236, 0.236, 0, 0.0001}, {2.0, 0.223, 0.223, 0.105, 0.0007},
                                    {4.3, 0.222, 0.370, 0.023, 0.0010}};

// Predicted us of the unsplit kernel of 17 - 64 rows of n > kWide columns.
inline double wide_time(uint32_t rows, uint32_t k, uint32_t n, int wb, uint32_t cus) {
  const uint32_t bn = small_tile_columns(rows, n);
  int kind = rows <= 24 ? 0 : 1;
  if (small_tiles_pay(rows, n)) kind = rows > 32 ? 4 : (bn == 64 ? 2 : 3);
  const WideCost& c = wb == 1 ? kWideCost8[kind] : kWideCost16[kind];
  const double wmb = static_cast<double>(n) * k * wb * 1e-6;
  return c.c0 + (plan_cdiv(n, bn) <= cus ? c.step1 : c.step2) * plan_cdiv(k, 64u) + (c.weight + c.row * rows) * wmb;
}

// Whether 65 - 256 rows of an int8 product leave 32-row skinny tiles with split
// K (w8a16.hip), which re-read the int8 weights per tile mostly from L2,
// faster than unsplit tiles: tiny grids (fewer than 32 64 x 64 tiles: 1.5B
// k/v at 96 - 256 rows, 6.4 vs 10.5 us) and narrow outputs (n < 2048) up to
// 128 rows (1.5B down, 128 rows 30.7 vs 34.3 us).  Wider outputs and more
// rows re-read too much (7B down, 96 rows 105.6 vs 82.8 us).
inline bool w8_skinny_pays(uint32_t rows, uint32_t n) {
  return rows <= 256 && (plan_cdiv(n, 64u) * plan_cdiv(rows, 64u) < 32 || (rows <= 128 && n < 2048));
}

struct SplitPlan {
  int tile;     // index into the split table; < 0: the unsplit kernels are faster
  int splits;   // K ranges, >= 2
  double cost;  // predicted us
  int direct;   // more than 64 rows: the fastest unsplit tile (index into kW8Cost / kL16Cost)
};

// The fastest split tile and count for [rows, k] x [n, k] (wb: bytes per
// weight), against the fastest unsplit kernel at that size.  One workgroup
// per CU: S = CUs / tiles, no more than 32, at least 4 K steps each, every
// range with work.  Splitting has to win 3% and 1.5 us in the prediction (an
// eager call also pays the second launch and the workspace on the host); on
// wide outputs at 17 - 64 rows also 1% against the kernels that run there.
// (The stream kernel's line alone split 86 int8 gate/up shapes that small
// tiles run faster: 3584 -> 18944, 64 rows 30.8 us unsplit, 39.3 split; 1536
// -> 8960, 64 rows 10.9 and 12.1.  What still splits: 5120 -> 13824 int8, 24
// rows 28.0 -> 22.1, 64 rows 28.7 -> 26.0; 18944 -> 9000, 64 rows int8 83.8
// -> 48.4, 16-bit 98.2 -> 67.4.  Over the sweep of 465 sizes the old line
// split, two of the slower ones still do (0.8% and 1.4%; they were slower by up
// to 2.0x), and 31 of the faster ones no longer do, by up to 13%.)
inline SplitPlan split_plan(uint32_t rows, uint32_t k, uint32_t n, int wb, uint32_t cus) {
  const TileCost* sc = wb == 1 ? kSplitCost8 : kSplitCost16;
  const double wmb = static_cast<double>(n) * k * wb * 1e-6;
  SplitPlan best{-1, 1, 1e30, 0};
  if (rows <= 16) return best;
  double direct, wide = kNoLaunch;
  if (rows <= 64) {
    const int cls = rows <= 24 ? 0 : (rows <= 32 ? 1 : (rows <= 48 ? 2 : 3));
    const double* st = wb == 1 ? kStreamCost8[cls] : kStreamCost16[cls];
    direct = st[0] + st[1] * wmb;
    if (n > kWide) wide = 0.99 * wide_time(rows, k, n, wb, cus);
  } else {
    const TilePlan unsplit = wb == 1 ? plan_tiles(kW8Cost, rows, n, k, wmb, cus, false)
                                     : plan_tiles(kL16Cost, rows, n, k, wmb, cus, false);
    best.direct = unsplit.shape;
    direct = unsplit.cost;
    // 32-row skinny tiles, one K chain per workgroup (896 k 5.5 us, 1536 k
    // 6.3, 3584 k 10.7, 4864 k 15.5)
    if (wb == 1 && w8_skinny_pays(rows, n) && 3.0 + 0.0023 * k < direct) direct = 3.0 + 0.0023 * k;
  }
  const double margin = 0.97 * direct < direct - 1.5 ? 0.97 * direct : direct - 1.5;
  const double limit = margin < wide ? margin : wide;
  // 16-bit weight rows a multiple of 8 KiB apart, read by several ranges at
  // once: 1.05 - 1.3x the prediction at 4096, 8192 and 12288 columns on wide
  // outputs (4096 -> 16384, 17 rows: 28.3 predicted, 35.7 us measured)
  const double strided = wide < kNoLaunch && wb == 2 && k % 4096 == 0 ? 1.15 : 1.0;
  const uint32_t steps = plan_cdiv(k, 64u);
  for (int t = 0; t < SPLIT_TILES; ++t) {
    const double fixed = sc[t].c0 + sc[t].weight * wmb;
    if (fixed >= limit) continue;
    // 64 bits: the size query takes any rows and n below 2^31, beyond what a launch may hold
    const uint64_t all = static_cast<uint64_t>(plan_cdiv(rows, static_cast<uint32_t>(sc[t].bm))) *
                         plan_cdiv(n, static_cast<uint32_t>(sc[t].bn));
    if (2 * all > cus) continue;
    const uint32_t tiles = static_cast<uint32_t>(all);
    uint32_t s = cus / tiles;
    if (s > 32) s = 32;
    if (s > steps / 4) s = steps / 4;
    if (s < 2) continue;
    const uint32_t per = plan_cdiv(steps, s);
    s = plan_cdiv(steps, per);
    if (s < 2) continue;
    const double c = strided * (fixed + sc[t].step * per + sc[t].part * 8e-6 * s * rows * n);
    if (c < best.cost && c < limit) best = SplitPlan{t, static_cast<int>(s), c, best.direct};
  }
  return best;
}

inline int64_t split_bytes(const SplitPlan& sp, int64_t rows, int64_t n) {
  return sp.tile < 0 ? 0 : static_cast<int64_t>(sizeof(float)) * sp.splits * rows * n;
}

// ------------------------------------------------------------- the launches

template <typename T, int BK, int WGM, int WGN, int FM, int FN, int S>
int split_gemm_cfg(const Params& p0, hipStream_t s) {
  using C = Cfg<T, BK, F32, WGM, WGN, FM, FN, EPI_PART, S>;
  static_assert(C::LDS <= 160 * 1024, "LDS per workgroup");
  Params p = p0;
  p.tiles_m = (p.rows + C::BM - 1) / C::BM;
  p.tiles_n = (p.n + C::BN - 1) / C::BN;
  p.group_m = p.tiles_m < 4 ? p.tiles_m : 4;
  void* args[] = {&p};
  return hip_status(
      hipLaunchKernel(reinterpret_cast<const void*>(tiled_gemm<T, BK, F32, WGM, WGN, FM, FN, EPI_PART, S, 1>),
                      dim3(static_cast<unsigned>(p.tiles_m * p.tiles_n * p.splits)), dim3(C::BLOCK), args, 0, s),
      "split-K launch");
}

// Both passes of plan sp; p holds the caller's operands and epilogue.
template <typename T, int BK, typename TO, int EPI>
int split_k_launch(Params p, const SplitPlan& sp, float* part, hipStream_t s) {
  p.part = part;
  p.splits = sp.splits;
  int st = MI355_ERR_UNSUPPORTED;
  switch (sp.tile) {
    case 0: st = split_gemm_cfg<T, BK, 1, 4, 1, 1, 4>(p, s); break;
    case 1: st = split_gemm_cfg<T, BK, 2, 2, 1, 1, 4>(p, s); break;
    case 2: st = split_gemm_cfg<T, BK, 1, 4, 2, 1, 4>(p, s); break;
    case 3: st = split_gemm_cfg<T, BK, 2, 4, 2, 1, 3>(p, s); break;
    case 4: st = split_gemm_cfg<T, BK, 2, 4, 4, 2, 2>(p, s); break;
    default: set_error("split-K: no tile %d", sp.tile);
  }
  if (st != MI355_OK) return st;
  const bool vec = p.n % 4 == 0 && p.os % 4 == 0 && aligned16(p.out);
  const int64_t threads = static_cast<int64_t>(p.rows) * p.n / (vec ? 4 : 1);
  void* args[] = {&p};
  const void* kern = vec ? reinterpret_cast<const void*>(split_k_reduce<TO, EPI, 4>)
                         : reinterpret_cast<const void*>(split_k_reduce<TO, EPI, 1>);
  return hip_status(hipLaunchKernel(kern, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), args, 0, s),
                    "split-K reduction launch");
}

}  // namespace tiled
}  // namespace mi355
