// How the decode GEMV (fh_gemv.hip) splits a call: its items, and the K slices its workgroups' waves take.
#pragma once
#include <algorithm>
#include "fh_epilogue.h"

namespace fh {

// rows a lane has in flight at once, by format and batch rows (about 4 KiB of weight a wave and run at batch 1)
__host__ __device__ constexpr int gemv_group(bool four, int b) { return (b <= 2 ? 4 : b <= 4 ? 2 : 1) * (four ? 2 : 1); }

// threads a workgroup at most: 16 waves for one row, 8 for more (whose partial sums need the registers)
__host__ __device__ constexpr int gemv_threads(int b) { return b == 1 ? 1024 : 512; }

// The K slices: W waves a workgroup, the least power of 2 giving about 16384 waves in all (64 a CU on 256 CUs, in
// turns), at most 8 for more than one row (their launch bound is 512 threads, so that the rows' partial sums stay in
// registers: bound to 1024 threads they spilled, and batch 8 of an 8B step took 35.6 ms instead of 6.5), at most 16 for bfp4
// and 8 for bfp8 at one row (a bfp8 wave needs ~100 registers at two runs an item, so a 16-wave workgroup fills a CU alone
// and the grid runs in lock-step rounds: on MI355X the 8B shapes' bfp8 gate_up 31.7 us at 16, 25.9 at 8; bfp4's down 11.0
// at 16, 11.4 at 8), and at most one a group of U loads of 64 rows a lane, whole or not: such a slice is one memory latency
// long, and shorter ones only add waves to start and sums to meet. (K 576 in bfp8, groups of 256 rows, in 2, 3 and 5 slices:
// qkv 4.5, 3.9, 4.6 us, gate_up 4.4, 3.7, 4.4, SmolLM's step 700, 627, 684; in bfp4, groups of 512, in 2 and 5: gate_up 4.2,
// 5.5; 1536 x 576 in bfp4 in 2, 3 and 12: 3.8, 3.2, 4.8; 2048 x 2048 in 4 and 16: 3.7, 5.7.)
struct GemvPlan { int W, rows, P, most, items; };
inline GemvPlan gemv_plan(int64_t K, int64_t N, int fmt, int kind, int batch) {
  GemvPlan p;
  p.P = (kind == FH_EP_SILU_GATE || kind == FH_EP_ROPE_KV) ? 2 : 1;  // as epilogue_args sets MatArgs::P
  p.most = p.P == 1 ? 8 : 4;
  p.items = (int)(N / 16 / p.P);
  const int b = batch < p.most ? batch : p.most;
  const int unit = 64 * gemv_group(fmt == FH_BFP4, b);
  const int64_t units = (K + unit - 1) / unit;
  const int64_t most = std::min<int64_t>(fmt == FH_BFP4 ? 16 : 8, gemv_threads(b) / 64);
  int64_t W = 1;
  while (W < most && W * p.items < 16384) W *= 2;
  W = std::min(W, units);
  int64_t rows = (K + W - 1) / W;
  rows = (rows + 63) / 64 * 64;
  p.W = (int)((K + rows - 1) / rows);
  p.rows = (int)rows;
  return p;
}

}  // namespace fh
