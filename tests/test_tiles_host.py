"""The matmul kernels' index rules and plans, compiled for the host from the headers the kernels include (no GPU needed)."""
import subprocess
import pytest
from ferrite_amd import build

RAGGED = r'''
#include "fh_gemm.h"
#include <cstdio>
template <int RUNS> static int walk(const fh::MatArgs& a) {  // every pair lane of every tile, as the epilogues take them
  int past = 0;
  for (int tn = 0; tn < (a.items + RUNS / 2 - 1) / (RUNS / 2); ++tn)
    for (int p = 0; p < RUNS / 2; ++p) {
      const int64_t run = fh::tile_run<RUNS>(a, tn, p);
      for (int j = 0; j < 16; ++j) {
        const fh::RopePair r = fh::rope_pair(a.head_dim, a.heads + a.kv_heads, run, j);
        const bool in = r.d >= 0 && r.d < a.head_dim / 2 && r.d1 == r.d + a.head_dim / 2;
        if (run < 0 ? r.turn : !in || r.h < 0) { printf("run %ld j %d: h %d d %d turn %d\n", (long)run, j, r.h, r.d, r.turn); return -1; }
        if (run >= 0 && ((int64_t)r.h * a.head_dim + r.d != run * 16 + j || r.turn != (r.h < a.heads + a.kv_heads))) return -2;
      }
      past += run < 0;
    }
  return past;
}
int main(int, char** v) {
  fh::MatArgs a = {};
  a.heads = atoi(v[1]); a.kv_heads = atoi(v[2]); a.head_dim = atoi(v[3]);
  a.P = 2; a.pair_half = a.head_dim / 32; a.N = (int64_t)(a.heads + 2 * a.kv_heads) * a.head_dim; a.items = (int)(a.N / 32);
  const int got[3] = {walk<8>(a), walk<12>(a), walk<16>(a)};
  for (int g : got) if (g < 0) return 1;
  printf("%d %d %d\n", got[0], got[1], got[2]);
}
'''


def program(d, text):
  (d / "t.hip").write_text(text)
  subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-w", "-I", str(build.CSRC),
                  "-I", str(build.HERE.parent / "include"), str(d / "t.hip"), "-o", str(d / "t")], check=True)
  return d / "t"


@pytest.fixture(scope="module")
def ragged(tmp_path_factory):
  return program(tmp_path_factory.mktemp("tiles"), RAGGED)


@pytest.mark.parametrize("heads,kv,hd", [(9, 3, 64), (1, 1, 32), (4, 1, 32), (5, 2, 64), (1, 1, 96), (3, 1, 160), (32, 8, 128)])
def test_rope_pairs_past_the_weight_read_no_table(ragged, heads, kv, hd):
  """A tile's pairs past the weight (SmolLM's qkv: 30 pairs in tiles of 4, 6 and 8) turn nothing, whatever their lane:
  at place 0 a turn there would read the 16 values before the tables."""
  r = subprocess.run([str(ragged), str(heads), str(kv), str(hd)], capture_output=True, text=True)
  assert r.returncode == 0, r.stdout
  pairs = (heads + 2 * kv) * hd // 32
  assert [int(x) for x in r.stdout.split()] == [-pairs % 4, -pairs % 6, -pairs % 8]


GEMV = r'''
#include "fh_gemv.h"
#include <cstdio>
int main() {
  for (int fmt : {FH_BFP8, FH_BFP4})
    for (int kind : {FH_EP_STORE, FH_EP_SILU_GATE})
      for (int batch : {1, 2, 3, 4, 5, 8, 9})
        for (int64_t K : {1, 63, 64, 65, 256, 257, 512, 576, 1024, 1025, 1536, 2048, 2816, 4096, 14336})
          for (int64_t N : {32, 576, 960, 4096, 49152, 1 << 22}) {
            const fh::GemvPlan p = fh::gemv_plan(K, N, fmt, kind, batch);
            printf("%d %d %d %ld %ld %d %d %d %d %d\n", fmt, kind, batch, (long)K, (long)N, p.W, p.rows, p.P, p.most, p.items);
          }
}
'''


def test_gemv_slices_are_whole_load_groups(tmp_path):
  """The GEMV's K slices cover K once, in whole 64 rows, none empty, within its workgroups' waves, and never more of them
  than the groups of loads a wave keeps in flight: shorter ones made bfp4 calls of few items up to twice as slow."""
  from ferrite_amd import lib
  lines = [list(map(int, l.split())) for l in subprocess.run([str(program(tmp_path, GEMV))], capture_output=True, text=True, check=True).stdout.splitlines()]
  assert len(lines) == 2 * 2 * 7 * 15 * 6
  for fmt, kind, batch, K, N, W, rows, P, most, items in lines:
    b = min(batch, most)
    assert P == (2 if kind == lib.EP_SILU_GATE else 1) and items == N // 16 // P
    assert rows % 64 == 0 and (W - 1) * rows < K <= W * rows and 1 <= W <= (16 if b == 1 and fmt == lib.BFP4 else 8)
    group = 64 * (4 if b <= 2 else 2 if b <= 4 else 1) * (2 if fmt == lib.BFP4 else 1)
    assert W <= -(-K // group), (fmt, kind, batch, K, N, W)


PACK = r'''
#include "fh_pack.h"
#include <cstdio>
int main() {
  for (int64_t K : {1, 4, 7, 8, 15, 16, 64, 4096, 4194240, 4194241})
    for (int64_t runs : {1ll, 8192ll, 16384ll, 131072ll, 1ll << 26, (1ll << 28) - 1, 1ll << 28, 1ll << 29})
      printf("%ld %ld %d\n", (long)K, (long)runs, fh::pack_in_tiles(K, runs));
}
'''


def test_packing_in_tiles_where_it_is_the_faster(tmp_path):
  """Packing along N in tiles of 64 rows: not of fewer than 8 rows, whose tiles are mostly idle threads (1 row 1.8 times as
  slow as a thread a block), and never past what a grid holds, which a thread a block takes (2^32 blocks)."""
  out = subprocess.run([str(program(tmp_path, PACK))], capture_output=True, text=True, check=True).stdout.splitlines()
  got = {(int(k), int(r)): t == "1" for k, r, t in (l.split() for l in out)}
  for (K, runs), tiles in got.items():
    assert tiles == (K >= 8 and K * runs >= 131072 and (runs + 15) // 16 * 256 < 2 ** 32 and -(-K // 64) < 65536), (K, runs)


PLAN = r'''
#include "fh_gemm.h"
#include <cstdio>
int main(int c, char** v) {
  for (int i = 1; i + 2 < c; i += 3) {
    const fh::GemmPlan p = fh::gemm_lds_plan(atoll(v[i]), atoll(v[i + 1]), atoll(v[i + 2]), 0, true);
    printf("%d %d\n", p.bm, p.splits);
  }
}
'''


def test_the_tiled_matmuls_tests_take_the_plans_they_name(tmp_path):
  """The shapes of the tiled matmul's GPU tests have the tiles and the parts of K that they are there for, and both tiles
  are there whole and in parts."""
  from test_gpu_16_gemm_lds import HD, PLANS, ROPES
  want = [(s, p) for s, p in PLANS.items()] + [((M, K, (h + 2 * kv) * HD), p) for (M, K, h, kv), p in ROPES.items()]
  args = [str(x) for s, _ in want for x in s]
  out = subprocess.run([str(program(tmp_path, PLAN)), *args], capture_output=True, text=True, check=True).stdout.splitlines()
  assert [tuple(map(int, l.split())) for l in out] == [p for _, p in want]
  for plans in (PLANS, ROPES): assert {(bm, s > 1) for bm, s in plans.values()} >= {(128, False), (128, True), (256, True)}
  assert (256, 1) in PLANS.values()


CHOICE = r'''
#include "fh_gemm.h"
#include <cstdio>
int main(int c, char** v) {  // M K N pairs: the kernel that bf16 rows take, with K in parts allowed
  for (int i = 1; i + 3 < c; i += 4) {
    fh::MatArgs a = {};
    a.M = atoll(v[i]); a.K = atoll(v[i + 1]); a.N = atoll(v[i + 2]); a.P = atoi(v[i + 3]); a.items = (int)(a.N / 16 / a.P);
    const fh::GemmPlan p = fh::gemm_lds_plan(a.M, a.K, a.N, 0, true);
    const fh::GemmWide w = fh::gemm_wide_plan(a, 256);
    if (p.us <= fh::gemm_wide_us(w, a.K, 256)) printf("lds%d\n", p.bm);
    else printf("pp%d\n", w.wn);
  }
}
'''


def test_the_faster_kernel_past_a_round(tmp_path):
  """Past one round of tiles a prompt's matmuls take the kernel and tile that measured fastest: each line one that another
  rule got wrong (us measured in lds128, lds256 and one round of the wide tiles). lds128: 128-row tiles, two a CU."""
  want = {(4096, 2048, 3072, 2): "lds128",   # 81, 97, 100 (192 columns)
          (3000, 4096, 6144, 2): "lds128",   # 220, 233
          (800, 4096, 28672, 2): "lds128",   # 273, 287
          (1600, 2048, 11264, 2): "lds128",  # 118, 126
          (1200, 2048, 11264, 2): "lds256",  # 88, 85
          (2048, 1024, 5632, 2): "lds128",   # 46, 56, 61
          (2048, 4096, 28672, 2): "lds256",  # 597, 533
          (4096, 4096, 6144, 2): "lds256",   # 268, 248
          (1400, 4096, 6144, 2): "pp3",      # 138, 138, 130
          (2048, 4096, 6144, 2): "pp3",      # 151, 143, 142
          (2300, 14336, 4096, 1): "pp3",     # 393 with K in parts, 326
          (3000, 14336, 4096, 1): "pp4",     # 433 with K in parts, 398
          (4096, 14336, 4096, 1): "pp4",     # 580, 498, 469
          (4096, 4096, 4096, 1): "lds256",   # 154, 178
          (2048, 14336, 4096, 1): "lds256"}  # one round: 238
  exe = program(tmp_path, CHOICE)
  out = subprocess.run([str(exe), *(str(x) for s in want for x in s)], capture_output=True, text=True, check=True).stdout.split()
  assert dict(zip(want, out)) == want


KEYS = r'''
#include "fh_prefill.h"
#include <cstdio>
int main(int c, char** v) {
  for (int i = 1; i + 3 < c; i += 4) printf("%d\n", fh::prefill_splits_keys(atoi(v[i]), atoi(v[i + 1]), atoi(v[i + 2]), atoll(v[i + 3]), 256));
}
'''


def test_prompt_keys_split_where_it_is_the_faster(tmp_path):
  """A short prompt's keys are split among a workgroup's waves where that gains in bf16 and does not lose in a block float,
  by one rule for all formats (us whole and split, in bf16, then in bfp8)."""
  want = {(100, 32, 128, 300): 1, (64, 32, 128, 1900): 1, (64, 32, 128, 4000): 1, (300, 32, 128, 0): 0,  # 51 30; 140 97 bfp8; past a round 13 18
          (64, 32, 128, 0): 0, (64, 32, 128, 64): 0, (33, 1, 128, 33): 0,  # one tile 5.2 7.1; two 8.4 8.8, 10.5 13.2; 10.0 12.2 bfp8
          (320, 1, 128, 0): 0, (200, 1, 128, 64): 0, (320, 1, 128, 1): 1,  # five: 17.1 15.4, 16.4 19.6; 17.0 18.3 bfp8; six
          (2, 9, 64, 64): 0, (96, 9, 64, 64): 1, (320, 9, 64, 0): 1,       # 7.6 8.1 bfp8; 10.1 8.8 bfp8; five: 12.9 11.8 bfp8
          (1, 300, 64, 5000): 0}
  out = subprocess.run([str(program(tmp_path, KEYS)), *(str(x) for k in want for x in k)], capture_output=True, text=True, check=True).stdout.split()
  assert dict(zip(want, map(int, out))) == want
