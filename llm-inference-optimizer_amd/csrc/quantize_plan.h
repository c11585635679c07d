// Which kernel of quantize_int8.hip a call takes.  Host code.
#pragma once

#include <stdint.h>

namespace mi355 {

// A row of `packets` 16-byte packets (0: rows that are no whole aligned ones).
struct QuantPlan {
  int vpl;       // packets a lane holds; 0: the generic kernel
  bool block;    // the workgroup's waves share one row, else a wave per row and 4 rows per workgroup
  int threads;   // per workgroup
  int64_t grid;  // workgroups
};

// One wave per row up to 8 packets a lane, then up to 16 waves of 4, then of
// 8.  A launch holds less than 2^32 threads: with a workgroup per row that is
// fewer rows (at 192 threads 22 million) than with a wave per row (67
// million), so the generic kernel takes the others, as it takes longer rows.
inline QuantPlan quant_plan(int64_t n, int64_t packets) {
  const int64_t lane = (packets + 63) / 64;
  const QuantPlan generic{0, false, 256, (n + 3) / 4};
  if (lane < 1 || lane > 16 * 8) return generic;
  if (lane <= 8) return QuantPlan{static_cast<int>(lane), false, 256, (n + 3) / 4};
  const int vpl = lane <= 16 * 4 ? 4 : 8;
  const int threads = 64 * static_cast<int>((lane + vpl - 1) / vpl);
  if (n * threads >= int64_t{1} << 32) return generic;
  return QuantPlan{vpl, true, threads, n};
}

}  // namespace mi355
