"""The tiled matmul kernels' index rules, compiled for the host from the headers the kernels include (no GPU needed)."""
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
        const fh::RopePair r = fh::rope_pair(a, run, j);
        const bool in = r.d >= 0 && r.d < a.head_dim / 2 && r.d1 == r.d + a.head_dim / 2;
        if (!in || r.h < 0 || (run < 0 && r.turn)) { printf("run %ld j %d: h %d d %d turn %d\n", (long)run, j, r.h, r.d, r.turn); return -1; }
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


@pytest.fixture(scope="module")
def ragged(tmp_path_factory):
  d = tmp_path_factory.mktemp("tiles")
  (d / "t.hip").write_text(RAGGED)
  subprocess.run([build.hipcc(), "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-w", "-I", str(build.CSRC),
                  "-I", str(build.HERE.parent / "include"), str(d / "t.hip"), "-o", str(d / "t")], check=True)
  return d / "t"


@pytest.mark.parametrize("heads,kv,hd", [(9, 3, 64), (1, 1, 32), (4, 1, 32), (5, 2, 64), (1, 1, 96), (3, 1, 160), (32, 8, 128)])
def test_rope_pairs_past_the_weight_read_no_table(ragged, heads, kv, hd):
  """A tile's pairs past the weight (SmolLM's qkv: 30 pairs in tiles of 4, 6 and 8) turn nothing, whatever their lane:
  at place 0 a turn there would read the 16 values before the tables."""
  r = subprocess.run([str(ragged), str(heads), str(kv), str(hd)], capture_output=True, text=True)
  assert r.returncode == 0, r.stdout
  pairs = (heads + 2 * kv) * hd // 32
  assert [int(x) for x in r.stdout.split()] == [-pairs % 4, -pairs % 6, -pairs % 8]
