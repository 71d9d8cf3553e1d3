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

// gemm_tiles' kernel for bf16 rows whose K is whole steps of 64 (fh_gemm_lds.hip)
struct GemmPlan { int bm; int splits; double us; };  // rows a tile, K's parts, and the time expected of it
bool gemm_lds_takes(const MatArgs& a);
GemmPlan gemm_lds_plan(int64_t M, int64_t K, int64_t N, int experts, bool may_split);
size_t gemm_lds_bytes(const GemmPlan& p, int64_t M, int64_t N);  // the splits' partial sums
int gemm_lds(const MatArgs& a, const SkinnyMoe& g, int fmt, int experts, const GemmPlan& p, float* parts, hipStream_t s);

}  // namespace fh
