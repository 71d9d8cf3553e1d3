// The tiled matmul by a block-float weight for bf16 rows whose K is whole steps of 64 (a prompt's matmuls, a mixture's
// gathered experts): x straight from memory into LDS, the weight converted on its way there.
//
// A workgroup of 8 waves takes 128 TM rows by 128 columns (8 runs of 16, or 4 runs and their RoPE / SiLU·gate
// partners), each wave 32 TM rows by two blocks of 32 columns, the second 64 columns after the first: a pair's two runs,
// so that a lane holds both of a pair's sums and the epilogue runs on the accumulators where they are. K steps of 64:
// x's rows go into a ring of two or three LDS stages by global_load_lds_dwordx4 (no registers, no LDS write instructions; each
// lane's address places its 16 bytes in the swizzled row). The weight's rows come in registers,
// three steps ahead (a lane a run's row: 16 bytes of bfp8, 8 of bfp4, and its exponent; a wave's loads 1 KiB or 512 B in
// one piece), and go as 16 bf16 values, row-major as they lie, into one of two stages while the matrix cores work on
// the other; ds_read_b64_tr_b16 reads them K-contiguous (fh_skinny.hip's read), so nothing is transposed on the way in.
// A row's 16-byte pieces are XOR-swizzled by the row so that 16 rows' writes, and a transposed read's four, meet no bank
// twice. One workgroup barrier a step.
//
// The products are gemm_kernel's, in its order: the same bits. Split (K in parts, for tiles that do not fill the CUs): a
// workgroup adds up its part and leaves the sums, as its lanes hold them, in the workspace; split_sum_kernel adds a
// tile's parts in order and runs the epilogue.
#include "fh_gemm.h"

namespace fh {

constexpr int GL_RUNS = GL_BN / 16, GL_NW = 8;  // a tile's runs, a workgroup's waves
static_assert(GL_RUNS == GL_NW, "a wave a run of the weight");

typedef short gl_short4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) gl_short4* gl_lds_short4;
typedef const __attribute__((address_space(1))) uint32_t* gl_global;
typedef __attribute__((address_space(3))) uint32_t* gl_lds;

// A wave's 16 rows m0 .. by two blocks of 32 columns (columns wc and 64 + wc of the tile) through a's epilogue, from cs
// (LDS, this wave's own: [16][GL_LDC], a row's two blocks side by side). rs: the rows' 1/rms, or null for 1; place, crow:
// RoPE's places and cache rows of them (all in LDS). Short loops,
// not unrolled rows: a workgroup runs this once, at the pace its instructions arrive (unrolled over the accumulators the
// kernel was 90 KB of code, and a call of one K step took 13 us).
// EPI: which of the epilogues this is the code of (GL_PLAIN: a store of the sums alone), a kernel each: one kernel of all of
// them needs their registers together, and with 128 rows a tile, where two workgroups a CU leave 128 a lane, kept 80 to 140
// bytes a lane of scratch (the 8B gate_up at 300 rows 125 us with 80, 156 with 136).
constexpr int GL_LDC = 68;
enum { GL_SUMS, GL_SILU, GL_ROPE, GL_PLAIN };
template <int EPI>
__device__ __forceinline__ void block_epilogue(const MatArgs& a, const SkinnyMoe& g, const float* cs, int tn, int wc, int64_t m0,
                                               int64_t M, int64_t ybase, int lane, const float* rs, const int32_t* place,
                                               const int32_t* crow, int64_t y0 = 0) {
  const int kind = EPI == GL_PLAIN ? FH_EP_STORE : a.kind;
  if constexpr (EPI == GL_SUMS || EPI == GL_PLAIN) {  // FH_EP_STORE, FH_EP_RESIDUAL: a lane 4 columns of a row, 4 rows a pass
    const int q = lane & 15, c = 4 * q, lc = wc + (c & 31);
    const int64_t run = tile_run<GL_RUNS>(a, tn, 4 * (q >> 3) + (lc >> 4)), col = run * 16 + (lc & 15);
    const bool res = kind == FH_EP_RESIDUAL;
    const bool vec = !((a.ldy | y0) & 3) && !((uintptr_t)a.y & 15) && !(res && ((uintptr_t)a.residual & 15));
    float4 old[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // (the rows' loads before the first store, which may alias them)
      const float* p = a.residual + (ybase + min(m0 + (lane >> 4) + 4 * i, M - 1)) * a.ldy + col;
      old[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (res && run >= 0) old[i] = vec ? *(const float4*)p : make_float4(p[0], p[1], p[2], p[3]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = (lane >> 4) + 4 * i;
      const int64_t m = m0 + r, at = y0 + (ybase + m) * a.ldy + col;
      const bool ok = m < M && run >= 0;
      float4 v = *(const float4*)(cs + r * GL_LDC + c);
      if (rs) { v.x *= rs[r]; v.y *= rs[r]; v.z *= rs[r]; v.w *= rs[r]; }
      if (res) { v.x += old[i].x; v.y += old[i].y; v.z += old[i].z; v.w += old[i].w; }
      if (ok) {
        if (vec && !a.y_bf16) *(float4*)((float*)a.y + at) = v;
        else if (vec) *(uint2*)((uint16_t*)a.y + at) = make_uint2(bf16_rne_f(v.x) | bf16_rne_f(v.y) << 16, bf16_rne_f(v.z) | bf16_rne_f(v.w) << 16);
        else { store_out(a.y, a.y_bf16, at, v.x); store_out(a.y, a.y_bf16, at + 1, v.y); store_out(a.y, a.y_bf16, at + 2, v.z); store_out(a.y, a.y_bf16, at + 3, v.w); }
      }
      if (res && a.copy_bf16 && ok) { put_copy(a, m, col, v.x); put_copy(a, m, col + 1, v.y); put_copy(a, m, col + 2, v.z); put_copy(a, m, col + 3, v.w); }
      if (res && a.ssq_out) {  // (a run is 4 lanes' 4 columns: the pairs 8, 4, 2 and 1 columns apart, in that order)
        float s[4] = {v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) { s[k] += __shfl_xor(s[k], 2, 64); s[k] += __shfl_xor(s[k], 1, 64); }
        if (ok && !(q & 3)) a.ssq_out[m * (a.N / 16) + run] = (s[0] + s[2]) + (s[1] + s[3]);
      }
      if (EPI == GL_SUMS && kind == FH_EP_STORE && a.argmax_parts) {
        float bv = v.x;
        int bc = (int)col;
        if (v.y > bv) { bv = v.y; bc = (int)col + 1; }
        if (v.z > bv) { bv = v.z; bc = (int)col + 2; }
        if (v.w > bv) { bv = v.w; bc = (int)col + 3; }
#pragma unroll
        for (int k = 2; k >= 1; k >>= 1) {
          const float ov = __shfl_xor(bv, k, 64);
          const int oc = __shfl_xor(bc, k, 64);
          if (ov > bv || (ov == bv && oc < bc)) { bv = ov; bc = oc; }
        }
        if (ok && !(q & 3)) a.argmax_parts[m * (a.N / 16) + run] = make_int2(__float_as_int(bv), bc);
      }
    }
    return;
  }
  // the pairs: a lane a column of the first run (its partner in the second block), 2 rows a pass; a run is 16 lanes
  const int c = lane & 31, j = lane & 15;
  const int64_t run = tile_run<GL_RUNS>(a, tn, (wc + c) >> 4), c0 = run * 16 + j;
  if constexpr (EPI == GL_SILU) {
    float sc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sc[i] = g.scale_rows ? g.row_w[ybase + min(m0 + (lane >> 5) + 2 * i, M - 1)] : 1.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = (lane >> 5) + 2 * i;
      const float s = rs ? rs[r] : 1.f;
      if (m0 + r < M && run >= 0)
        store_out(a.y, a.y_bf16, (ybase + m0 + r) * a.ldy + c0, silu(cs[r * GL_LDC + c] * s) * (cs[r * GL_LDC + 32 + c] * s) * sc[i]);
    }
    return;
  }
  const int hd = a.head_dim;
  const auto [h, d, d1, turn] = rope_pair(hd, a.heads + a.kv_heads, run, j);  // (turn: x cos + (-x2, x1) sin, models/llama.py:92-93)
  float tab[2][4][4];  // 4 rows' table values, and the next 4's: all loads before the first store, which may alias them
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    float* v = tab[u >> 2][u & 3];
    v[0] = v[1] = 1.f;
    v[2] = v[3] = 0.f;
    if (turn) {
      const int64_t at = rope_place(a, place[(lane >> 5) + 2 * u]) * hd;
      v[0] = a.cos_tab[at + d]; v[1] = a.cos_tab[at + d1];
      v[2] = a.sin_tab[at + d]; v[3] = a.sin_tab[at + d1];
    }
  }
#pragma unroll 1
  for (int i0 = 0; i0 < 8; i0 += 4) {  // (a loop of two: the put into a cache is long)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = (lane >> 5) + 2 * (i0 + u);
      const int64_t m = m0 + r;
      if (m >= M || run < 0) continue;
      const float s = rs ? rs[r] : 1.f;
      float x0 = cs[r * GL_LDC + c] * s, x1 = cs[r * GL_LDC + 32 + c] * s;
      if (turn) {
        const float* v = tab[0][u];
        const float t0 = x0 * v[0] - x1 * v[2], t1 = x1 * v[1] + x0 * v[3];
        x0 = t0; x1 = t1;
      }
      if (h < a.heads) {
        float* q = (float*)a.y + m * a.ldy + (int64_t)h * hd;
        q[d] = x0; q[d1] = x1;
      } else {
        cache_put(a, h - a.heads, crow[r], d, d1, j, x0, x1);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int k = 0; k < 4; ++k) tab[0][u][k] = tab[1][u][k];
  }
}

// A wave's blocks' values of 16 rows (values r = 8 half .. + 7 of each block: rows 16 half .. + 15) into cs
__device__ __forceinline__ void block_to_lds(float* cs, const floatx16 (&v)[2], int half, int lane) {
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)
    if (hh == half)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 8; ++r) cs[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * GL_LDC + 32 * j + (lane & 31)] = v[j][8 * hh + r];
}

// MODE 0: K whole; 1: a part of K, its sums left in `parts`; 2: a part of K whose outputs go g.split_y elements after the
// part before's (a store's only: whoever reads them adds them up)
template <bool FOUR, int TM, int MODE, int EPI>
__global__ __launch_bounds__(64 * GL_NW, TM == 2 ? 2 : 4) void gemm_lds_kernel(MatArgs a, SkinnyMoe g, int tiles_m, int tiles_n, int splits,
                                                                              float* parts) {
  constexpr bool SPLIT = MODE != 0;
  constexpr int BM = 128 * TM, NS = TM == 2 || SPLIT ? 2 : 3;
  constexpr int AB = BM * GL_BK * 2, BB = GL_BK * GL_BN * 2;
  constexpr int IA = AB / 1024 / GL_NW;  // a wave's loads of x a step (1 KiB, 8 rows each)
  constexpr int WL = 2;                  // and of the weight: a lane a row of its run, and the row's exponent
  constexpr int RB = FOUR ? 8 : 16;
  using Row = typename std::conditional<FOUR, uint2, uint4>::type;
  __shared__ __attribute__((aligned(16))) char a0[AB];
  __shared__ __attribute__((aligned(16))) char a1[AB];
  __shared__ __attribute__((aligned(16))) char a2[NS == 3 ? AB : 16];
  __shared__ __attribute__((aligned(16))) char b0[BB];
  __shared__ __attribute__((aligned(16))) char b1[BB];

  // this workgroup's expert, part of K and tile: tiles (each its parts one after another) go to the XCDs in contiguous ranges,
  // in groups of 8 row tiles
  int64_t M = a.M, ybase = 0;
  const uint8_t* wmant = a.mant;
  const uint8_t* wexps = a.exps;
  int id = blockIdx.x, tiles = tiles_m * tiles_n;
  if (g.counts) {
    const int e = blockIdx.y;
    M = min((int64_t)g.counts[e], a.M);
    ybase = (int64_t)e * a.M;
    wmant += e * g.expert_mant;
    wexps += e * g.expert_exps;
    tiles_m = (int)((M + BM - 1) / BM);
    tiles = tiles_m * tiles_n;
    const int q = (tiles * splits + 7) / 8;
    if (id >= 8 * q) return;
    id = (id % 8) * q + id / 8;
    if (id >= tiles * splits) return;
  } else if (tiles * splits % 8 == 0) {
    id = (id % 8) * (tiles * splits / 8) + id / 8;
  }
  const int part = SPLIT ? id % splits : 0;  // (a tile's parts on one XCD: their sums meet in its L2)
  if (SPLIT) id /= splits;
  const int per_group = 8 * tiles_n, first_m = id / per_group * 8, gm = min(tiles_m - first_m, 8);
  const int tm = first_m + (id % per_group) % gm, tn = (id % per_group) / gm;
  const int64_t m0 = (int64_t)tm * BM;
  const int all = (int)(a.K / GL_BK);
  const int first = SPLIT ? (int)((int64_t)all * part / splits) : 0;
  const int steps = (SPLIT ? (int)((int64_t)all * (part + 1) / splits) : all) - first;

  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // x: load i of this wave fills rows 8 (wave IA + i) .. + 7 of a stage, lane l the l-th 16 bytes: row l / 8, piece l % 8,
  // which holds piece (l % 8) ^ (row / 2 % 8) of the row (rows past M read the last one)
  const uint16_t* px[IA];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int r = 8 * (wave * IA + i) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int64_t m = min(m0 + r, M - 1);
    const int64_t row = g.counts ? (g.x_rows ? (int64_t)g.x_rows[ybase + m] : ybase + m) : m;
    px[i] = (const uint16_t*)a.x + row * a.ldx + (int64_t)first * GL_BK + 8 * c;
  }
  auto load_x = [&](char* s, int step) {
#pragma unroll
    for (int i = 0; i < IA; ++i)
      __builtin_amdgcn_global_load_lds((gl_global)(px[i] + (int64_t)min(step, steps - 1) * GL_BK), (gl_lds)(s + (wave * IA + i) * 1024), 16, 0, 0);
  };
  // the weight: run `wave` of the tile, row `lane` of the step (a run past the weight reads the first; its columns are not
  // stored)
  const int64_t nb = tile_run<GL_RUNS>(a, tn, wave), w0 = (nb < 0 ? 0 : nb) * a.K + (int64_t)first * GL_BK + lane;
  const uint8_t* pm = wmant + w0 * RB;
  const uint8_t* pe = wexps + w0;
  Row wm[2];
  uint32_t we[2];
  auto load_w = [&](int step, int set) {
    const int64_t k = (int64_t)min(step, steps - 1) * GL_BK;
    wm[set] = *(const Row*)(pm + k * RB);
    we[set] = pe[k];
  };
  auto swz = [](int k) { return 4 * (k & 3) + ((k >> 2) & 3); };  // row k's XOR on a piece's place
  auto store_w = [&](char* s, int set) {
    float f[16];
    magnitudes(wm[set], f);
    const float sc = ldexpf(1.f, (int)we[set] - 133);
    uint32_t w[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) w[q] = pack_bf16_exact(f[2 * q] * sc, f[2 * q + 1] * sc);
    char* row = s + lane * GL_BN * 2;
    *(uint4*)(row + ((2 * wave ^ swz(lane)) << 4)) = make_uint4(w[0], w[1], w[2], w[3]);
    *(uint4*)(row + (((2 * wave + 1) ^ swz(lane)) << 4)) = make_uint4(w[4], w[5], w[6], w[7]);
  };

  floatx16 acc[TM][2];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int wr = (wave >> 1) * 32 * TM, wc = (wave & 1) * 32;
  const bool live = m0 + wr < M;  // (else none of this wave's rows are there: it only loads for the others)
  const int fr = lane & 31, fh8 = lane >> 5;
  const int rm = (lane >> 2) & 3, rq = lane & 3, rg = (lane >> 4) & 1;
  auto compute = [&](const char* sa, const char* sb) {
    if (TM == 1 && MODE != 1 && !live) return;  // (an expert's 128-row tile is often a third empty)
#pragma unroll
    for (int kk = 0; kk < GL_BK; kk += 16) {
      bf16x8 fa[TM], fb[2];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int r = wr + 32 * i + fr;
        fa[i] = *(const bf16x8*)(sa + r * GL_BK * 2 + (((kk / 8 + fh8) ^ ((r >> 1) & 7)) << 4));
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int k = kk + 8 * fh8 + rm, c = (64 * j + wc + 16 * rg + 4 * rq) >> 3;
        union { gl_short4 s[2]; bf16x8 v; } u;
        u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gl_lds_short4)(sb + k * GL_BN * 2 + ((c ^ swz(k)) << 4) + 8 * (rq & 1)));
        u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gl_lds_short4)(sb + (k + 4) * GL_BN * 2 + ((c ^ swz(k + 4)) << 4) + 8 * (rq & 1)));
        fb[j] = u.v;
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
  };

  // Step s: wait for this wave's loads of x's stage s (issued after them, with two stages: the weight of s + 2; with three:
  // the weight of s + 1, x of s + 1 and the weight of s + 2), for its LDS writes and its reads of the last step, meet the
  // others; then x of s + NS - 1 goes out, the weight of s + 1 into its stage, the weight of s + 3 out, and the products
  // (the compiler interleaves the conversion with them). Past the last step the loads read it again, into stages and
  // registers that nobody reads.
#define GL_A(i) ((i) % NS == 0 ? a0 : (i) % NS == 1 ? a1 : a2)
#define GL_B(i) ((i) % 2 == 0 ? b0 : b1)
  load_x(a0, 0);
  load_w(0, 0);
  asm volatile("" ::: "memory");
  if (NS == 3) load_x(a1, 1);
  asm volatile("" ::: "memory");
  load_w(1, 1);
  store_w(b0, 0);
  load_w(2, 0);
  constexpr int TURN = NS == 2 ? 2 : 6;  // (both stage counts divide it)
  for (int q = 0; q < steps; q += TURN) {
#pragma unroll
    for (int i = 0; i < TURN; ++i) {
      if (q + i >= steps) break;
      constexpr int W = NS == 3 ? IA + 2 * WL : WL;  // vmcnt(W) lgkmcnt(0)
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0x0070 | (W & 15) | (W >> 4) << 14);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      load_x(GL_A(i + NS - 1), q + i + NS - 1);
      asm volatile("" ::: "memory");
      store_w(GL_B(i + 1), (i + 1) & 1);
      load_w(q + i + 3, (i + 1) & 1);
      compute(GL_A(i), GL_B(i));
    }
  }
#undef GL_A
#undef GL_B
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070);  // (no load into LDS outlives its workgroup)
  if (MODE == 1) {
    if (!live) return;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      float* p = parts + (((int64_t)(part * tiles + id) * GL_NW + wave) * TM + i) * 2048 + lane;
      if (m0 + wr + 32 * i < M)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) p[(16 * j + r) * 64] = acc[i][j][r];
    }
    return;
  }
  __syncthreads();  // the stages are free: each wave's outputs, 16 rows at a time, in a part of x's of its own
  constexpr int CW = 16 * GL_LDC * 4, WPA = AB / CW;
  static_assert(MODE == 1 || (NS + 2) * WPA >= GL_NW, "the outputs' place");
  float* cs = (float*)((wave < WPA ? a0 : wave < 2 * WPA ? a1 : wave < 3 * WPA ? (NS == 3 ? a2 : b1) : b0) + wave % WPA * CW);
  float* rs_s = (float*)b0;  // where the weight was: the rows' 1/rms, and RoPE's places and cache rows
  int32_t* rows_s = (int32_t*)b0 + BM;
  if (MODE == 0 && (a.ssq_in || EPI == GL_ROPE)) {
    if (a.ssq_in)
#pragma unroll 1
      for (int r = 16 * wave; r < BM; r += 16 * GL_NW) row_scales16(a, rs_s + r, m0 + r, lane);
    if (EPI == GL_ROPE && t < BM) stage_rope_rows(a, rows_s, BM, t, min(m0 + t, M - 1));
    __syncthreads();
  }
#pragma unroll 1
  for (int u = 0; u < 2 * TM && m0 + wr + 16 * u < M; ++u) {
#pragma unroll
    for (int ii = 0; ii < TM; ++ii)  // (the accumulators' indices stay constants)
      if (ii == u >> 1) block_to_lds(cs, acc[ii], u & 1, lane);
    wave_lds_order();
    block_epilogue<EPI>(a, g, cs, tn, wc, m0 + wr + 16 * u, M, ybase, lane, MODE == 0 && a.ssq_in ? rs_s + wr + 16 * u : nullptr,
                              rows_s + wr + 16 * u, rows_s + BM + wr + 16 * u, MODE == 2 ? part * g.split_y : 0);
    wave_lds_order();
  }
}

// The split tiles' sums: a wave 16 rows by 2 x 32 columns of a tile (half of a wave's block there), its parts added in order,
// four parts' loads in flight at a time, then the epilogue. Bound by reading the parts once (splits x 4 bytes an output),
// from the L2 of the XCD that wrote them (o at 200 rows in bfp4, both launches: 30.6 -> 24.7 us against parts dealt to
// the XCDs part by part).
template <int TM, int EPI>
__global__ __launch_bounds__(256) void split_sum_kernel(MatArgs a, SkinnyMoe g, int tiles_m, int tiles_n, int splits, const float* parts) {
  __shared__ float rs_s[4][16];
  __shared__ int32_t rows_s[4][32];
  __shared__ __attribute__((aligned(16))) float cs_s[4][16 * GL_LDC];
  const int64_t M = a.M;
  const int tiles = tiles_m * tiles_n;
  // (workgroups dealt to the XCDs in contiguous ranges, as the tiles' were: a tile's parts are in this XCD's L2)
  const int nb = gridDim.x, blk = nb % 8 == 0 ? (int)(blockIdx.x % 8) * (nb / 8) + (int)blockIdx.x / 8 : (int)blockIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, u = blk * 4 + w;  // unit u: (tile, wave, i, half)
  const int half = u & 1, i = (u >> 1) % TM, wave = (u >> 1) / TM % GL_NW, id = (u >> 1) / (TM * GL_NW);
  if (id >= tiles) return;
  const int per_group = 8 * tiles_n, first_m = id / per_group * 8, gm = min(tiles_m - first_m, 8);
  const int tm = first_m + (id % per_group) % gm, tn = (id % per_group) / gm;
  const int64_t m0 = (int64_t)tm * 128 * TM + ((wave >> 1) * TM + i) * 32 + 16 * half;
  if (m0 >= M) return;
  float* rs = rs_s[w];
  float* cs = cs_s[w];
  int32_t* rows = rows_s[w];  // (this wave's own rows)
  if (a.ssq_in) row_scales16(a, rs, __builtin_amdgcn_readfirstlane((int)m0), lane);  // (m0 < 2^31: below 2^23 tiles)
  if (EPI == GL_ROPE && lane < 16) stage_rope_rows(a, rows, 16, lane, min(m0 + lane, M - 1));
  const int64_t stride = (int64_t)tiles * GL_NW * TM * 2048;
  const float* p = parts + (((int64_t)id * GL_NW + wave) * TM + i) * 2048 + 512 * half + lane;
  float acc[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int s = 0; s < splits; s += 4) {
    float v[4][16];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int r = 0; r < 16; ++r) v[k][r] = p[min(s + k, splits - 1) * stride + (r & 7) * 64 + (r >> 3) * 1024];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += s + k < splits ? v[k][r] : 0.f;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) cs[(8 * ((r & 7) >> 2) + 4 * (lane >> 5) + (r & 3)) * GL_LDC + 32 * (r >> 3) + (lane & 31)] = acc[r];
  wave_lds_order();
  block_epilogue<EPI>(a, g, cs, tn, (wave & 1) * 32, m0, M, 0, lane, a.ssq_in ? rs : nullptr, rows, rows + 16);
}

bool gemm_lds_takes(const MatArgs& a) {
  return a.kind != FH_EP_PROGRAM && a.x_bf16 && !a.x_tiles && !a.y_tiles && !a.copy_tiles && !a.norm_w && a.K % GL_BK == 0 && !((uintptr_t)a.x & 15) && a.ldx % 8 == 0;
}

int gemm_lds(const MatArgs& a, const SkinnyMoe& g, int fmt, int experts, const GemmPlan& p, float* parts, hipStream_t s) {
  const int64_t tm = (a.M + p.bm - 1) / p.bm, all = gemm_lds_grid(a, p), tn = all / p.splits / tm;
  if (!gemm_lds_fits(a, p)) return fail(FH_EUNSUP, "fh_gemm_bfp: too many tiles");
  if (p.splits > 1 && !g.split_y && (!parts || g.counts)) return fail(FH_EINVAL, "fh_gemm_bfp: K in parts needs a place for their sums");
  const dim3 grid((unsigned)(g.counts ? (all + 7) / 8 * 8 : all), g.counts ? experts : 1), block(64 * GL_NW);
#define GL_RUN(F, TM, MODE, EPI) hipLaunchKernelGGL((gemm_lds_kernel<F, TM, MODE, EPI>), grid, block, 0, s, a, g, (int)tm, (int)tn, p.splits, parts)
#define GL_SUM(TM, EPI) hipLaunchKernelGGL((split_sum_kernel<TM, EPI>), dim3((unsigned)(tm * tn * 4 * TM)), dim3(256), 0, s, a, g, (int)tm, (int)tn, p.splits, (const float*)parts)
#define GL(F, TM) do { \
    if (p.splits > 1 && TM == 1 && g.split_y) GL_RUN(F, 1, 2, GL_PLAIN); \
    else if (p.splits > 1) { \
      GL_RUN(F, TM, 1, GL_PLAIN); \
      if (a.P == 1) GL_SUM(TM, GL_SUMS); \
      else if (a.kind == FH_EP_SILU_GATE) GL_SUM(TM, GL_SILU); \
      else GL_SUM(TM, GL_ROPE); \
    } else if (a.P == 1) GL_RUN(F, TM, 0, GL_SUMS); \
    else if (a.kind == FH_EP_SILU_GATE) GL_RUN(F, TM, 0, GL_SILU); \
    else GL_RUN(F, TM, 0, GL_ROPE); } while (0)
  if (p.bm == 256) { if (fmt == FH_BFP4) GL(true, 2); else GL(false, 2); }
  else if (fmt == FH_BFP4) GL(true, 1);
  else GL(false, 1);
#undef GL
#undef GL_SUM
#undef GL_RUN
  return check_launch("fh_gemm_bfp");
}

}  // namespace fh
