// The lazy Tensor's matmul of plain operands on the matrix cores: C[b] = program(A[b] @ B[b]), A [M][K] and B [K][N]
// each bf16 or fp32 (ferrite/tensor.py:443-485 with a bf16 or fp32 B). bf16 x bf16 products, exact in fp32, summed in
// fp32; an fp32 operand goes in as two bf16 parts, hi (its value rounded to nearest even) and lo (what hi leaves,
// rounded), and the sum is hi@hi + hi@lo + lo@hi (lo@lo, about 2^-16 of the rest, left out), ferrite's bf16x3
// (tensor.py:674-689): about 16 significant bits of each operand.
//
// A workgroup of WR x WC waves computes a tile of BM x BN outputs in K steps of BK, each wave TM x TN blocks of 32 x 32
// (v_mfma_f32_32x32x16_bf16). Both operands lie in LDS as they lie in memory, A [BM][BK] and B [BK][BN], the 16-byte
// pieces of a row XOR-swizzled so that neither writes nor fragment reads meet in a bank (64 banks: b128 reads measured
// at 229 of 256 bytes a clock, 128 with an 8-row swizzle, 32 with none). A's fragments are read 16 bytes a lane, B's
// through ds_read_b64_tr_b16 (in each 16-lane group, lane 4 m + q addresses row m, columns 4 q .. 4 q + 3, and lane j
// receives column j of the four rows), K-contiguous as the matrix cores take them, so B needs no transposing writes.
// The products come in the same order in every kernel and tile: the same bits.
//
// matmul_lds_kernel: bf16 operands of whole 16-byte pieces and K steps. Rows go straight from memory into a ring of NS
// LDS stages (global_load_lds_dwordx4: no registers, no LDS write instructions), the swizzle in each lane's address;
// one workgroup barrier a step. What bounds it is the step's latency, not a stream: 4096^3 runs at ~1060 TFLOP/s in
// tiles of 128 x 256 (129 us; 2730 us before, in 64 x 64 tiles of bounds-checked element loads), with the ring two
// steps deep; 256 x 256 tiles in two stages 960-1060 and fewer of them; 128 x 128 tiles in four stages, where the wide
// ones leave CUs idle (2048^3: 570 -> 800 TFLOP/s).
//
// matmul_kernel: everything else (fp32 operands, any shape, stride and alignment): through registers into two LDS
// stages. A thread's loads of the step after next are in flight while the matrix cores work on this one: 8 consecutive
// elements of a row each, at any even alignment; rows at odd strides, and the last step's part past K, an element at a
// time.
//
// The epilogue takes each wave's blocks through its own part of LDS, 32 rows at a time, so that a row's outputs leave
// in 16-byte stores. The fused elementwise program runs there in place, 4 rows a pass of the wave: an element at a time
// its decoding is what these tiles' 8 waves a CU wait for (of 9 ops: fp32 4096 x 16 x 4096 413 us, so 237, which 64 x 64
// tiles of 20 KiB of LDS, 8 waves a SIMD, took too; bf16 2048^3 125 us, so 57; one op 47, so 31).
#include "fh_program.h"

namespace fh {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 mm_bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float mm_floatx16;
typedef short mm_short4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) mm_short4* mm_lds_short4;

struct MmArgs {
  const void* a; int64_t sa, lda;
  const void* b; int64_t sb, ldb;
  int64_t M, K, N;
  void* c; int c_dtype; int64_t sc, ldc;
  int avec, bvec;     // rows of A / B at 4-byte alignment: 16-byte loads
  int cvec;           // C's rows at 16-byte alignment: 16-byte stores
  int tiles_m, tiles_n;
};

struct __attribute__((packed, aligned(4))) MmWords4 { uint32_t x, y, z, w; };  // 16 bytes at 4-byte alignment

// 8 consecutive elements as loaded: 4 words of bf16, or 8 of fp32
template <bool F32>
struct MmPiece {
  uint32_t w[F32 ? 8 : 4];
  __device__ void vec(const char* p) {
#pragma unroll
    for (int i = 0; i < (F32 ? 2 : 1); ++i) {
      const MmWords4 v = ((const MmWords4*)p)[i];
      w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
    }
  }
  __device__ void some(const char* p, int n) {  // the first n elements (n <= 0: none), the rest 0
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (F32) w[j] = j < n ? ((const uint32_t*)p)[j] : 0u;
      else {
        const uint32_t h = j < n ? ((const uint16_t*)p)[j] : 0u;
        w[j >> 1] = (j & 1) ? w[j >> 1] | h << 16 : h;
      }
    }
  }
  __device__ uint4 hi() const {
    if (!F32) return make_uint4(w[0], w[1], w[2], w[3]);
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = bf16_rne(w[2 * i & 7]) | bf16_rne(w[(2 * i + 1) & 7]) << 16;
    return make_uint4(o[0], o[1], o[2], o[3]);
  }
  __device__ uint4 lo() const {
    uint32_t o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t v = w[F32 ? i : 0];
      o[i] = bf16_rne_f(__uint_as_float(v) - bf16_to_f(bf16_rne(v)));
    }
    return make_uint4(o[0] | o[1] << 16, o[2] | o[3] << 16, o[4] | o[5] << 16, o[6] | o[7] << 16);
  }
};

// The workgroup's tile. Tiles go to the XCDs in contiguous ranges (workgroups are dealt to them round-robin), in groups of
// 8 row tiles, so that an XCD's L2 keeps the rows and columns its tiles share.
__device__ inline void matmul_place(const MmArgs& m, int& tm, int& tn) {
  const int tiles = m.tiles_m * m.tiles_n;
  int id = blockIdx.x;
  if (tiles % 8 == 0) id = (id % 8) * (tiles / 8) + id / 8;
  const int per_group = 8 * m.tiles_n, first_m = id / per_group * 8, gm = min(m.tiles_m - first_m, 8);
  tm = first_m + (id % per_group) % gm;
  tn = (id % per_group) / gm;
}

// A wave's outputs, TM blocks of 32 rows by TN of 32 columns from (r0, col0), through cs (32 rows of 32 TN + 4 floats)
template <int TM, int TN, bool PROG>
__device__ inline void matmul_epilogue(const MmArgs& m, const fh_program& p, const mm_floatx16 (&acc)[TM][TN], float* cs, int64_t bi,
                                       int64_t r0, int64_t col0, int lane) {
  constexpr int CLD = 32 * TN + 4;
  const int fr = lane & 31, fh8 = lane >> 5;
  // value r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of a block
  const int64_t cbase = bi * m.sc;
  for (int i = 0; i < TM; ++i) {
    wave_lds_order();
#pragma unroll
    for (int ii = 0; ii < TM; ++ii) {  // (the accumulators' indices stay constants)
      if (ii != i) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) cs[(8 * (r >> 2) + 4 * fh8 + (r & 3)) * CLD + 32 * j + fr] = acc[ii][j][r];
    }
    wave_lds_order();
    const int64_t row0 = r0 + 32 * i;
    if (PROG) {
      constexpr int R = 64 / (32 * TN), E = TM * TN > 4 ? 2 : 4;  // rows a pass of the wave, passes at a time (2: registers)
      const int c = lane % (32 * TN), rl = lane / (32 * TN);
      const int64_t rows = m.M - row0, col = min(col0 + c, m.N - 1);
      for (int rr = 0; rr < 32 && rr < rows; rr += E * R) {  // (whole waves: places past M or N read the last there is)
        const int r = rr + rl;
        float v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = cs[(r + e * R) * CLD + c];
        prog_eval_rows<E>(p, v, bi, row0 + r, R, m.M - 1, col);
#pragma unroll
        for (int e = 0; e < E; ++e) cs[(r + e * R) * CLD + c] = v[e];
      }
      wave_lds_order();
    }
    const bool inside = row0 + 32 <= m.M && col0 + 32 * TN <= m.N;
    if (m.cvec && inside && m.c_dtype != FH_I32) {
      if (m.c_dtype == FH_BF16) {
        constexpr int L = 4 * TN;  // lanes a row, 8 columns each
#pragma unroll
        for (int q = 0; q < 32 * L / 64; ++q) {
          const int r = (lane + 64 * q) / L, c = 8 * (lane % L);
          const float4 u = *(const float4*)(cs + r * CLD + c), v = *(const float4*)(cs + r * CLD + c + 4);
          *(uint4*)((uint16_t*)m.c + cbase + (row0 + r) * m.ldc + col0 + c) =
              make_uint4(bf16_rne_f(u.x) | bf16_rne_f(u.y) << 16, bf16_rne_f(u.z) | bf16_rne_f(u.w) << 16,
                         bf16_rne_f(v.x) | bf16_rne_f(v.y) << 16, bf16_rne_f(v.z) | bf16_rne_f(v.w) << 16);
        }
      } else {
        constexpr int L = 8 * TN;  // lanes a row, 4 columns each
#pragma unroll
        for (int q = 0; q < 32 * L / 64; ++q) {
          const int r = (lane + 64 * q) / L, c = 4 * (lane % L);
          *(float4*)((float*)m.c + cbase + (row0 + r) * m.ldc + col0 + c) = *(const float4*)(cs + r * CLD + c);
        }
      }
    } else {
      for (int e = lane; e < 32 * 32 * TN; e += 64) {
        const int r = e / (32 * TN), c = e % (32 * TN);
        const int64_t row = row0 + r, col = col0 + c;
        if (row < m.M && col < m.N) prog_store(m.c, m.c_dtype, cbase + row * m.ldc + col, cs[r * CLD + c]);
      }
    }
  }
}

typedef const __attribute__((address_space(1))) uint32_t* mm_global;
typedef __attribute__((address_space(3))) uint32_t* mm_lds;

// bf16, rows 16-byte aligned, N in whole pieces, K in whole steps
template <int WR, int WC, int TM, int TN, int NS, bool PROG>
__global__ __launch_bounds__(WR * WC * 64, 1) void matmul_lds_kernel(MmArgs m, fh_program p) {
  constexpr int NW = WR * WC, BM = WR * TM * 32, BN = WC * TN * 32, BK = 64, CA = BK / 8, CB = BN / 8;
  constexpr int AB = BM * BK * 2, STAGE = AB + BK * BN * 2;
  constexpr int IA = AB / 1024 / NW, IB = BK * BN * 2 / 1024 / NW, PER = IA + IB;  // a wave's loads of 1 KiB a stage
  constexpr int CW = 32 * (32 * TN + 4) * 4;
  static_assert(NS >= 3 && NS <= 4 && NW * CW <= 3 * STAGE && CB >= 16, "stages");
  // (an array a stage: the compiler then sees that a stage's reads do not wait for the others' loads)
  __shared__ __attribute__((aligned(16))) char s0[STAGE];
  __shared__ __attribute__((aligned(16))) char s1[STAGE];
  __shared__ __attribute__((aligned(16))) char s2[STAGE];
  __shared__ __attribute__((aligned(16))) char s3[NS > 3 ? STAGE : 16];
  const int64_t bi = blockIdx.z;
  int tm_, tn_;
  matmul_place(m, tm_, tn_);
  const int64_t m0 = (int64_t)tm_ * BM, n0 = (int64_t)tn_ * BN;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);

  // where piece c of row r lies (matmul_kernel's, at BK 64 and BN 128 or more)
  auto at_a = [&](int r, int c) { return r * BK * 2 + ((c ^ ((r >> 1) & 7)) << 4); };
  auto at_b = [&](int r, int c) { return r * BN * 2 + ((c ^ (4 * (r & 3))) << 4); };
  // a wave's load i writes 64 pieces in a line, lane l the l-th: row u / C, place u % C of the stage; rows past M read the
  // last, columns past N the last piece (their products are not stored)
  const uint16_t* pa[IA];
  const uint16_t* pb[IB];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int u = (wave * IA + i) * 64 + lane, r = u / CA, c = (u % CA) ^ ((r >> 1) & 7);
    pa[i] = (const uint16_t*)m.a + bi * m.sa + min(m0 + r, m.M - 1) * m.lda + 8 * c;
  }
#pragma unroll
  for (int i = 0; i < IB; ++i) {
    const int u = (wave * IB + i) * 64 + lane, r = u / CB, c = (u % CB) ^ (4 * (r & 3));
    pb[i] = (const uint16_t*)m.b + bi * m.sb + (int64_t)r * m.ldb + min(n0 + 8 * c, m.N - 8);
  }
  auto load = [&](char* s, int64_t k0) {
#pragma unroll
    for (int i = 0; i < IA; ++i) __builtin_amdgcn_global_load_lds((mm_global)(pa[i] + k0), (mm_lds)(s + (wave * IA + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < IB; ++i) __builtin_amdgcn_global_load_lds((mm_global)(pb[i] + k0 * m.ldb), (mm_lds)(s + AB + (wave * IB + i) * 1024), 16, 0, 0);
  };

  mm_floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int wr = wave / WC * TM * 32, wc = wave % WC * TN * 32;
  const int fr = lane & 31, fh8 = lane >> 5;
  const int tm = (lane >> 2) & 3, tq = lane & 3, tg = (lane >> 4) & 1;
  auto compute = [&](const char* s) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      mm_bf16x8 fa[TM], fb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i] = *(const mm_bf16x8*)(s + at_a(wr + 32 * i + fr, kk / 8 + fh8));
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int k = kk + 8 * fh8 + tm, c = (wc + 32 * j + 16 * tg + 4 * tq) >> 3;
        union { mm_short4 s[2]; mm_bf16x8 v; } u;
        u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((mm_lds_short4)(s + AB + at_b(k, c) + 8 * (tq & 1)));
        u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((mm_lds_short4)(s + AB + at_b(k + 4, c) + 8 * (tq & 1)));
        fb[j] = u.v;
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
  };

  // Step s: wait for this wave's loads of its stage (those of the NS - 2 stages after it may be in flight) and for its
  // reads of the last one, meet the others, send the loads of step s + NS - 1 into the stage just read, then the
  // products. Past the last step the loads read it again, into stages that nobody reads.
#define MM_STAGE(i) ((i) % NS == 0 ? s0 : (i) % NS == 1 ? s1 : (i) % NS == 2 ? s2 : s3)
  const int64_t steps = m.K / BK;
#pragma unroll
  for (int i = 0; i < NS - 1; ++i) load(MM_STAGE(i), min((int64_t)i, steps - 1) * BK);
  for (int64_t q = 0; q < steps; q += NS) {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      if (q + i >= steps) break;
      constexpr int W = (NS - 2) * PER;  // vmcnt(W) lgkmcnt(0)
      static_assert(W < 64, "vmcnt's range");
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0x0070 | (W & 15) | (W >> 4) << 14);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      load(MM_STAGE(i + NS - 1), min(q + i + NS - 1, steps - 1) * BK);
      compute(MM_STAGE(i));
    }
  }
#undef MM_STAGE
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070);  // (every load into LDS has landed before the outputs go there)
  __syncthreads();
  // each wave's outputs in a part of a stage of its own
  constexpr int WPS = STAGE / CW;  // waves a stage holds
  static_assert(WPS >= 1 && (NW + WPS - 1) / WPS <= 3, "the outputs' place");
  char* cs = (wave / WPS == 0 ? s0 : wave / WPS == 1 ? s1 : s2) + wave % WPS * CW;
  matmul_epilogue<TM, TN, PROG>(m, p, acc, (float*)cs, bi, m0 + wr, n0 + wc, lane);
}

// Any operands
template <int WR, int WC, int TM, int TN, int BK, bool AF, bool BF, bool PROG>
__global__ __launch_bounds__(WR * WC * 64, 1) void matmul_kernel(MmArgs m, fh_program p) {
  constexpr int NT = WR * WC * 64, BM = WR * TM * 32, BN = WC * TN * 32;
  constexpr int CA = BK / 8, CB = BN / 8;  // 16-byte pieces a row of A's and B's tiles
  constexpr int PA = BM * CA / NT, PB = BK * CB / NT;  // pieces a thread
  constexpr int AB = BM * BK * 2, BB = BK * BN * 2;  // bytes of a part
  constexpr int STAGE = AB * (AF ? 2 : 1) + BB * (BF ? 2 : 1);
  constexpr int CLD = 32 * TN + 4, CW = 32 * CLD * 4;  // a wave's 32 rows of outputs
  constexpr int LDS = 2 * STAGE > WR * WC * CW ? 2 * STAGE : WR * WC * CW;
  static_assert(BM * CA % NT == 0 && BK * CB % NT == 0 && CA >= 4 && CB >= 8, "whole pieces");
  __shared__ __attribute__((aligned(16))) char smem[LDS];

  const int64_t bi = blockIdx.z;
  int tm_, tn_;
  matmul_place(m, tm_, tn_);
  const int64_t m0 = (int64_t)tm_ * BM, n0 = (int64_t)tn_ * BN;

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t K = m.K;
  constexpr int EA = AF ? 4 : 2, EB = BF ? 4 : 2;
  // A: piece t + NT i of the tile, row (t / CA) + (NT / CA) i, k 8 (t % CA) ..; rows past M read the last one
  const int ar = t / CA, ac = 8 * (t % CA);
  const char* ap[PA];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int64_t r = m0 + ar + NT / CA * i;
    ap[i] = (const char*)m.a + (bi * m.sa + (r < m.M ? r : m.M - 1) * m.lda + ac) * EA;
  }
  // B: piece t + NT i, k row (t / CB) + (NT / CB) i, columns 8 (t % CB) ..
  const int br = t / CB, bc = 8 * (t % CB);
  const int nleft = (int)min((int64_t)8, m.N - n0 - bc);  // columns of this thread's pieces that are there
  const char* bp = (const char*)m.b + (bi * m.sb + (int64_t)br * m.ldb + n0 + bc) * EB;
  const int64_t bstep = (int64_t)(NT / CB) * m.ldb * EB;

  MmPiece<AF> ra[PA];
  MmPiece<BF> rb[PB];
  // the fast load: no bounds but the columns' (a piece at most 7 columns past N: the row after's first ones, in memory
  // as long as a row comes after; a piece past N the last even column)
  const char* bq = (const char*)m.b + (bi * m.sb + (int64_t)br * m.ldb + min(n0 + bc, (m.N - 1) & ~(int64_t)1)) * EB;
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int i = 0; i < PA; ++i) ra[i].vec(ap[i] + k0 * EA);
#pragma unroll
    for (int i = 0; i < PB; ++i) rb[i].vec(bq + k0 * m.ldb * EB + bstep * i);
  };
  // the careful one: an element at a time where a row's stride or a piece's end asks for it
  auto load_part = [&](int64_t k0) {
    const bool whole = k0 + BK <= K;
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      if (m.avec && whole) ra[i].vec(ap[i] + k0 * EA);
      else ra[i].some(ap[i] + k0 * EA, (int)min((int64_t)8, K - k0 - ac));
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const bool row = k0 + br + NT / CB * i < K;
      const char* q = bp + k0 * m.ldb * EB + bstep * i;
      if (m.bvec && row && nleft == 8) rb[i].vec(q);
      else rb[i].some(q, row ? nleft : 0);
    }
  };
  // where piece c of row r lies: A's rows swizzled by the 256 bytes of banks (256 / (2 BK) rows), so that a fragment's
  // rows, a row apart, meet no bank twice; B's so that the four k rows of a transposed read meet none
  constexpr int RWA = 128 / BK > 0 ? 128 / BK : 1;
  auto at_a = [&](int r, int c) { return r * BK * 2 + ((c ^ ((r / RWA) & (CA - 1))) << 4); };
  auto at_b = [&](int r, int c) { return r * BN * 2 + ((c ^ (CB >= 16 ? 4 * (r & 3) : 4 * ((r >> 1) & 1))) << 4); };
  auto store = [&](int stage) {
    char* s = smem + stage * STAGE;
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int at = at_a(ar + NT / CA * i, t % CA);
      *(uint4*)(s + at) = ra[i].hi();
      if (AF) *(uint4*)(s + AB + at) = ra[i].lo();
    }
    s += AB * (AF ? 2 : 1);
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int at = at_b(br + NT / CB * i, t % CB);
      *(uint4*)(s + at) = rb[i].hi();
      if (BF) *(uint4*)(s + BB + at) = rb[i].lo();
    }
  };

  mm_floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int wr = wave / WC * TM * 32, wc = wave % WC * TN * 32;
  const int fr = lane & 31, fh8 = lane >> 5;
  const int tm = (lane >> 2) & 3, tq = lane & 3, tg = (lane >> 4) & 1;  // the transposed read's row, quarter and 16 columns
  auto compute = [&](int stage) {
    const char* sa = smem + stage * STAGE;
    const char* sb = sa + AB * (AF ? 2 : 1);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      mm_bf16x8 ah[TM], al[TM], bh[TN], bl[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int at = at_a(wr + 32 * i + fr, kk / 8 + fh8);
        ah[i] = *(const mm_bf16x8*)(sa + at);
        if (AF) al[i] = *(const mm_bf16x8*)(sa + AB + at);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        // k rows kk + 8 fh8 + tm (then + 4), columns wc + 32 j + 16 tg + 4 tq ..
        const int k = kk + 8 * fh8 + tm, c = (wc + 32 * j + 16 * tg + 4 * tq) >> 3;
        const int at0 = at_b(k, c) + 8 * (tq & 1), at1 = at_b(k + 4, c) + 8 * (tq & 1);
        union { mm_short4 s[2]; mm_bf16x8 v; } u;
        u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((mm_lds_short4)(sb + at0));
        u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((mm_lds_short4)(sb + at1));
        bh[j] = u.v;
        if (BF) {
          u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((mm_lds_short4)(sb + BB + at0));
          u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((mm_lds_short4)(sb + BB + at1));
          bl[j] = u.v;
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
          if (BF) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
          if (AF) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
        }
    }
  };

  // Step s: the loads of step s + 1 go into the other stage, those of step s + 2 out, then the products. The last step's
  // loads (and every one of operands at odd strides) are careful ones; the others run in a loop of their own, where
  // nothing merges with them, so that each waits only for what it stores.
  const int64_t steps = (K + BK - 1) / BK;
  int cur = 0;
  for (int64_t s = -2; s < steps; ++s) {
    if (s == 0 && m.avec && m.bvec && m.N >= 8) {
      for (; s + 3 < steps; ++s) {
        store(1 - cur);
        load((s + 2) * BK);
        compute(cur);
        cur = 1 - cur;
        __syncthreads();
      }
    }
    if (s >= -1 && s + 1 < steps) store(s < 0 ? 0 : 1 - cur);
    if (s + 2 < steps) load_part((s + 2) * BK);
    if (s >= 0) { compute(cur); cur = 1 - cur; }
    __syncthreads();
  }

  matmul_epilogue<TM, TN, PROG>(m, p, acc, (float*)(smem + wave * CW), bi, m0 + wr, n0 + wc, lane);
}

// The kernel and tile for a product: the one whose rounds of workgroups take least, by a 64-k step's time of each in us
// as measured (alone on a CU / per tile with the chip full of them): tiles of 128 x 256 and 128 x 128 from LDS loads 1.0
// and 0.55 a round of one a CU; through registers bf16 256 x 256 1.9 a round, 128 x 128 0.84 / 0.71, 64 x 64 0.5 / 0.29,
// with an fp32 operand (two parts) 128 x 128 2.4 / 2.4, 64 x 64 1.3 / 0.9. (1024 x 4096 x 1024: 55 us in 64 tiles of 128 x
// 128, 33 in 256 of 64 x 64; 2048^3: 49 us in 64 x 64, 40 in 128 x 128, 21 from LDS loads.)
struct MmPlan { int bm, bn; bool lds; };
MmPlan matmul_plan(int64_t M, int64_t N, int64_t batch, bool f32, bool lds, int64_t cus) {
  static const struct { MmPlan p; double alone, full; bool f32; } plans[] = {
      {{128, 256, true}, 1.0, 1.0, false}, {{128, 128, true}, 0.55, 0.55, false},
      {{256, 256, false}, 1.9, 1.9, false}, {{128, 128, false}, 0.84, 0.71, false}, {{64, 64, false}, 0.5, 0.29, false},
      {{128, 128, false}, 2.4, 2.4, true}, {{64, 64, false}, 1.3, 0.9, true}};
  MmPlan best = {};
  double cost = 0;
  for (const auto& c : plans) {
    if (c.f32 != f32 || (c.p.lds && !lds)) continue;
    const int64_t per = (M + c.p.bm - 1) / c.p.bm * ((N + c.p.bn - 1) / c.p.bn), rounds = (per * batch + cus - 1) / cus;
    if (cost != 0 && per >= 1LL << 22) continue;  // (a grid's threads along x stay below 2^32)
    const double t = rounds * c.full > c.alone ? rounds * c.full : c.alone;
    if (cost == 0 || t < cost) { cost = t; best = c.p; }
  }
  return best;
}

}  // namespace fh

using namespace fh;

extern "C" int fh_matmul(const void* a, int a_dtype, int64_t a_batch_stride, int64_t lda, const void* b, int b_dtype,
                         int64_t b_batch_stride, int64_t ldb, int64_t batch, int64_t M, int64_t K, int64_t N,
                         const fh_program* program, void* c, int c_dtype, int64_t c_batch_stride, int64_t ldc,
                         void* stream) {
  if (!a || !b || !c) return fail(FH_EINVAL, "fh_matmul: null pointer");
  if ((a_dtype != FH_F32 && a_dtype != FH_BF16) || (b_dtype != FH_F32 && b_dtype != FH_BF16))
    return fail(FH_EINVAL, "fh_matmul: A and B are FH_F32 or FH_BF16");
  if (c_dtype != FH_F32 && c_dtype != FH_BF16 && c_dtype != FH_I32) return fail(FH_EINVAL, "fh_matmul: C is FH_F32, FH_BF16 or FH_I32");
  if (batch < 1 || M < 1 || K < 1 || N < 1) return fail(FH_EINVAL, "fh_matmul: batch, M, K and N at least 1");
  if (lda < K || ldb < N || ldc < N || a_batch_stride < 0 || b_batch_stride < 0 || c_batch_stride < 0)
    return fail(FH_EINVAL, "fh_matmul: a row stride below its row's length, or a negative batch stride");
  if (batch > 65535 || (M + 63) / 64 > 65535 || (N + 63) / 64 > (1LL << 31) - 1)
    return fail(FH_EUNSUP, "fh_matmul: batch or tiles past the grid's limits");
  if (program) {
    if (int rc = check_program("fh_matmul", program, true)) return rc;
  }
  // a program that only copies the sum is none
  const bool prog = program && !(program->n_ops == 1 && program->op[0] == FH_OP_COPY && program->a[0] == FH_OPND_ACC);
  MmArgs m = {a, a_batch_stride, lda, b, b_batch_stride, ldb, M, K, N, c, c_dtype, c_batch_stride, ldc};
  const bool af = a_dtype == FH_F32, bf = b_dtype == FH_F32;
  m.avec = !((uintptr_t)a & 3) && (af || (!(lda & 1) && !(a_batch_stride & 1)));
  m.bvec = !((uintptr_t)b & 3) && (bf || (!(ldb & 1) && !(b_batch_stride & 1)));
  const int64_t cv = c_dtype == FH_BF16 ? 8 : 4;
  m.cvec = !((uintptr_t)c & 15) && ldc % cv == 0 && c_batch_stride % cv == 0;
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    return n;
  }();
  const bool lds = !af && !bf && K % 64 == 0 && N % 8 == 0 && !((uintptr_t)a & 15) && !((uintptr_t)b & 15) && lda % 8 == 0 &&
                   ldb % 8 == 0 && a_batch_stride % 8 == 0 && b_batch_stride % 8 == 0;
  const MmPlan pl = matmul_plan(M, N, batch, af || bf, lds, cus);
  const int64_t tm = (M + pl.bm - 1) / pl.bm, tn = (N + pl.bn - 1) / pl.bn;
  if (tm * tn >= (pl.lds || pl.bm == 256 ? 1LL << 23 : 1LL << 24)) return fail(FH_EUNSUP, "fh_matmul: too many tiles");
  m.tiles_m = (int)tm; m.tiles_n = (int)tn;
  fh_program p = program ? *program : fh_program{};
  const dim3 grid((unsigned)(tm * tn), 1, (unsigned)batch);
  hipStream_t s = as_stream(stream);
#define MM(WR, WC, TM, TN, BK, A, B) \
  do { if (prog) hipLaunchKernelGGL((matmul_kernel<WR, WC, TM, TN, BK, A, B, true>), grid, dim3(WR * WC * 64), 0, s, m, p); \
       else hipLaunchKernelGGL((matmul_kernel<WR, WC, TM, TN, BK, A, B, false>), grid, dim3(WR * WC * 64), 0, s, m, p); } while (0)
#define MM_LDS(WR, WC, TM, TN, NS) \
  do { if (prog) hipLaunchKernelGGL((matmul_lds_kernel<WR, WC, TM, TN, NS, true>), grid, dim3(WR * WC * 64), 0, s, m, p); \
       else hipLaunchKernelGGL((matmul_lds_kernel<WR, WC, TM, TN, NS, false>), grid, dim3(WR * WC * 64), 0, s, m, p); } while (0)
#define MM_SIDES(A, B) do { if (pl.bm == 128) MM(2, 2, 2, 2, 32, A, B); else MM(2, 2, 1, 1, 64, A, B); } while (0)
  if (pl.lds) {
    if (pl.bn == 256) MM_LDS(2, 4, 2, 2, 3);
    else MM_LDS(4, 2, 1, 2, 4);
  } else if (af && bf) MM_SIDES(true, true);
  else if (af) MM_SIDES(true, false);
  else if (bf) MM_SIDES(false, true);
  else if (pl.bm == 256) MM(2, 4, 4, 2, 64, false, false);
  else if (pl.bm == 128) MM(2, 2, 2, 2, 64, false, false);
  else MM(2, 2, 1, 1, 64, false, false);
#undef MM_SIDES
#undef MM_LDS
#undef MM
  return check_launch("fh_matmul");
}
