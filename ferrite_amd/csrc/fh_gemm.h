// Shared by the tiled matmul kernels of a block-float weight (fh_gemm.hip, fh_gemm_lds.hip): the matrix cores' operand
// types, bf16 packing, and which run of the weight a tile's columns are.
#pragma once
#include "fh_epilogue.h"

namespace fh {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

__device__ inline uint32_t pack_bf16_exact(float lo, float hi) {  // both exact in bf16: the high halves
  // (the high halves of two floats whose low halves are 0: one byte permute, v_perm_b32)
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ inline uint32_t pack_bf16_rne(float lo, float hi) { return bf16_rne_f(lo) | (bf16_rne_f(hi) << 16); }

// the run a tile's local run lr (0 .. RUNS - 1) stands for, or -1 past the weight: RUNS runs of 16 columns a tile, or
// RUNS / 2 pairs (the first runs, then their partners)
template <int RUNS = 8>
__host__ __device__ inline int64_t tile_run(const MatArgs& a, int tn, int lr) {
  if (a.P == 1) {
    const int64_t nb = (int64_t)tn * RUNS + lr;
    return nb < a.N / 16 ? nb : -1;
  }
  const int64_t it = (int64_t)tn * (RUNS / 2) + lr % (RUNS / 2);
  if (it >= a.items) return -1;
  const int64_t nb0 = pair_first(it, a.pair_half);
  return lr < RUNS / 2 ? nb0 : nb0 + a.pair_half;
}

// 1/rms of 16 rows from m0 on (past the matrix: its last row's) into rs (LDS), from the sums of squares their maker left by
// runs of 16, by one wave: a row's sums lie along the lanes (a load of a wave is one piece of a row), 16 rows at once and two
// loads of each in flight, then the lanes' sums meet for all 16 rows together. (Two threads a row, each reading every other
// sum in turn, take 32 rows' lines a load: 30 us a 256-row tile of K 4096, or 57 by the waves that own the rows, against 5.)
__device__ __forceinline__ void row_scales16(const MatArgs& a, float* rs, int64_t m0, int lane) {
  const float* q = a.ssq_in + min(m0, a.M - 1) * a.ssq_parts;
  const int last = (int)min((int64_t)15, max((int64_t)0, a.M - 1 - m0));
  float v[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = 0.f;
#pragma unroll 1
  for (int i0 = 0; i0 < a.ssq_parts; i0 += 128) {
    const int i = i0 + lane, j = i + 64;
    const bool oki = i < a.ssq_parts, okj = j < a.ssq_parts;
    float u[2][16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t row = min(r, last) * a.ssq_parts;  // (a.ssq_parts < 2^27)
      u[0][r] = q[row + (oki ? i : 0)];
      u[1][r] = q[row + (okj ? j : 0)];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) { v[r] += oki ? u[0][r] : 0.f; v[r] += okj ? u[1][r] : 0.f; }
  }
  wave_reduce16(v);
  if (!(lane & 3)) rs[reduce16_index(lane)] = 1.0f / sqrtf(v[0] / (float)a.K + a.eps);
}

// row_scales16 of 32 rows: of few sums (a load a row) all 32 in flight at once, where a second pass would be half of the call
__device__ __forceinline__ void row_scales32(const MatArgs& a, float* rs, int64_t m0, int lane) {
  if (a.ssq_parts > 64) {
#pragma unroll 1
    for (int r = 0; r < 32; r += 16) row_scales16(a, rs + r, m0 + r, lane);
    return;
  }
  const float* q = a.ssq_in + min(m0, a.M - 1) * a.ssq_parts;
  const int last = (int)min((int64_t)31, max((int64_t)0, a.M - 1 - m0));
  const bool ok = lane < a.ssq_parts;
  float v[2][16];
#pragma unroll
  for (int r = 0; r < 32; ++r) v[r >> 4][r & 15] = q[min(r, last) * a.ssq_parts + (ok ? lane : 0)];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int r = 0; r < 16; ++r) v[h][r] = ok ? v[h][r] : 0.f;
    wave_reduce16(v[h]);
    if (!(lane & 3)) rs[16 * h + reduce16_index(lane)] = 1.0f / sqrtf(v[h][0] / (float)a.K + a.eps);
  }
}

// RoPE's per-row values for a tile's epilogue, staged in LDS: row ar's place and cache row (m: the row, clamped into the
// matrix)
__device__ inline void stage_rope_rows(const MatArgs& a, int32_t* rows_s, int bm, int ar, int64_t m) {
  rows_s[ar] = a.places[m];
  rows_s[bm + ar] = a.cache_rows[m];
}

// gemm_tiles' kernel for bf16 rows whose K is whole steps of 64 (fh_gemm_lds.hip): tiles of 128 columns in K steps of 64
constexpr int GL_BK = 64, GL_BN = 128;
struct GemmPlan { int bm; int splits; double us; };  // rows a tile, K's parts, and the time expected of it

// Rows a tile and K's parts: the least of a model of the call's time in us, its constants measured on a whole MI355X's 256
// CUs at 1K, 2K and 8B shapes (bfp8 and bfp4 alike). Up to a round of 128-row tiles two a CU, and K in parts: 8 a launch; a
// step of a 256-row tile 1.0 with a workgroup a CU, 1.15 a round of them with the chip full; of a 128-row tile 0.8 alone on a
// CU, 1.38 two a CU; K in parts, 6 more for the second launch and the parts written and read back at 6.5 TB/s. (Measured,
// 200 rows, 1 part -> the plan's: o 4096 x 4096 75 -> 26 us in 8, down 14336 x 4096 203 -> 45 in 8, qkv 4096 x 6144 67 -> 30 in
// 5; 1024 rows: o 72 -> 53 and down 214 -> 133 in 2; at 2048 rows every shape is fastest in one part.) K whole past that
// round: 128-row tiles fill a last round's places as others empty, so they pay for tiles and not for rounds, and each round's
// ramp and epilogue count beside its steps (7 a round of 256-row tiles, 1.3 of 128-row ones): 8B gate_up at 800
// rows 272 us in 1568 tiles of 128 rows, 287 in 896 of 256; 2048 x 11264 at 1600 118 and 126; at 2048 128 and 126. A
// gathered matmul (experts > 0), whose rows an expert the host does not know, takes 128-row tiles in one part.
inline GemmPlan gemm_lds_plan(int64_t M, int64_t K, int64_t N, int experts, bool may_split) {
  if (experts > 0) return {128, 1, 0};
  GemmPlan best = {};
  double cost = 0;
  const double full = (double)((M + 127) / 128 * ((N + GL_BN - 1) / GL_BN)) / 512;  // 128-row tiles, two a CU
  for (int bm = 256; bm >= 128; bm /= 2) {
    const int64_t tiles = (M + bm - 1) / bm * ((N + GL_BN - 1) / GL_BN), all = K / GL_BK;
    for (int s = 1; s <= (may_split ? 16 : 1) && (s == 1 || all / s >= 4); ++s) {
      const int64_t t = tiles * s;
      // (parts of at most 256 MB: past it the tiles are over a thousand already, and parts save the last round's rest alone)
      if (s > 1 && t * bm * GL_BN * 4 > (int64_t)256 << 20) break;
      double step;
      if (bm == 256) step = t <= 256 ? 1.0 : 1.15 * ((t + 255) / 256);
      else step = 1.38 * (t / 512) + (t % 512 == 0 ? 0 : t % 512 <= 256 ? 0.8 : 1.38);
      double us = 8 + (all + s - 1) / s * step + (s > 1 ? 6 + 8.0 * s * M * N / 6.5e6 : 0);
      if (s == 1 && full > 1) {
        if (bm == 256) us = t <= 256 ? 19 + 0.88 * all : 12 + (t + 255) / 256 * (7 + (double)all);
        else us = 1.3 * full + (full <= 2 ? 18.5 + (1.1 + 0.62 * full) * all : 20 + (0.16 + 1.23 * full) * all);
      }
      if (cost == 0 || us < cost) { cost = us; best = {bm, s, us}; }
    }
  }
  return best;
}

inline size_t gemm_lds_bytes(const GemmPlan& p, int64_t M, int64_t N) {
  return p.splits < 2 ? 0 : (size_t)p.splits * ((M + p.bm - 1) / p.bm) * ((N + GL_BN - 1) / GL_BN) * p.bm * GL_BN * 4;
}

// gemm_pp_kernel's 256-row tiles (fh_gemm.hip) of bf16 rows, 64 wn columns wide, 128, 192 or 256: the widest whose tiles fill
// the CUs' rounds (at most one round, or the last at least 7/8 full) and no narrower tile takes fewer rounds of as much work;
// none filling them (wn 0), gemm_kernel (qkv's 384 tiles of 2048 rows x 128 columns ran at 656 TFLOP/s against 712-750 for
// 128-row tiles two a CU)
struct GemmWide { int wn; int64_t tiles; };
inline GemmWide gemm_wide_plan(const MatArgs& a, int cus) {
  GemmWide w = {};
  int64_t best = 0;
  for (int wn = 2; wn <= 4; ++wn) {
    const int64_t tiles = (a.M + 255) / 256 * (a.P == 1 ? (a.N / 16 + 4 * wn - 1) / (4 * wn) : ((int64_t)a.items + 2 * wn - 1) / (2 * wn));
    const int64_t rounds = (tiles + cus - 1) / cus;
    const bool fills = tiles <= cus || tiles * 8 >= rounds * cus * 7;
    if (fills && (best == 0 || rounds * wn <= best)) { w = {wn, tiles}; best = rounds * wn; }
  }
  return w;
}
// The time expected of one round of its tiles of 192 or 256 columns, in us, by the share of the CUs they fill; no less than
// anything for narrower tiles or more rounds, which gemm_lds beats or meets within 4%. (Measured against gemm_lds: 8B qkv at 1536
// rows 131 us in 192 tiles and 138, at 2048 in 256 142 and 142; 14336 x 4096 at 2300 rows 326 in 198 and 393 with K in parts,
// at 4096 469 in 256 and 498; but 4096 x 4096 there 178 and 154, and 2048 x 3072 100 and 81.)
inline double gemm_wide_us(const GemmWide& w, int64_t K, int cus) {
  const double fill = (double)w.tiles / cus, steps = (double)(K / GL_BK);
  if (w.wn < 3 || w.tiles > cus) return 1e30;
  return w.wn == 3 ? 43 + (0.4 + 1.12 * fill) * steps : 50 + (0.6 + 1.28 * fill) * steps;
}

// its workgroups over a's rows (one expert's, gathered), and whether a grid of them is one that a launch holds (512 threads
// each, a grid's threads along x below 2^32)
inline int64_t gemm_lds_grid(const MatArgs& a, const GemmPlan& p) {
  return (a.M + p.bm - 1) / p.bm * (a.P == 1 ? (a.N / 16 + 7) / 8 : ((int64_t)a.items + 3) / 4) * p.splits;
}
inline bool gemm_lds_fits(const MatArgs& a, const GemmPlan& p) { return gemm_lds_grid(a, p) < 1LL << 23; }

bool gemm_lds_takes(const MatArgs& a);
int gemm_lds(const MatArgs& a, const SkinnyMoe& g, int fmt, int experts, const GemmPlan& p, float* parts, hipStream_t s);

}  // namespace fh
