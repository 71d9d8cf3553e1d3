"""The tiled matmul of bf16 rows whose x goes straight into LDS (fh_gemm_lds.hip): every epilogue at the edges of its
tiles of 128 and 256 rows, in one part of K against the kernel that fp32 rows take (the same bf16 products in the same order:
the same bits), and with K in parts within fp32 summation's error of that. Rows past M of x's buffer hold NaN: none may reach
a sum."""
import ctypes
import pytest
import torch
from ferrite_amd import llama as G

pytestmark = pytest.mark.gpu
HD = 64
# (M, K, N): the plan's rows a tile and parts of K. Both tiles, whole and in parts; one row or column block more or less than
# a tile; parts of unequal length (32 steps in 7, 64 in 13)
PLANS = {(65, 64, 16): (128, 1), (96, 192, 144): (128, 1), (127, 1536, 576): (128, 6), (128, 4096, 128): (128, 16), (129, 320, 2064): (128, 1),
         (200, 4096, 1024): (128, 16), (257, 576, 960): (128, 1), (300, 1024, 4096): (128, 1), (1000, 512, 6144): (256, 1),
         (129, 2048, 4112): (256, 7), (130, 4096, 2064): (256, 13), (257, 4096, 4096): (256, 4), (200, 1536, 6144): (256, 4)}
# the same for qkv matmuls: heads and kv heads of HD
ROPES = {(65, 64, 1, 1): (128, 1), (130, 576, 9, 3): (128, 1), (200, 576, 4, 1): (128, 1), (96, 4096, 5, 2): (128, 16), (300, 4096, 9, 3): (128, 10),
         (129, 2048, 33, 15): (128, 4), (257, 4096, 33, 15): (256, 4)}


def parts_bytes(lib, M, K, N, plan):
  """The workspace of the plan that the test is for."""
  bm, splits = plan
  n = lib.load().fh_gemm_workspace_bytes(M, K, N)
  assert n == (splits * -(-M // bm) * bm * -(-N // 128) * 128 * 4 if splits > 1 else 0)
  return n


def both(ops, lib, x, bw, make, out_shape, dtype, ws_bytes):
  """The call on fp32 rows (values of bf16), on bf16 rows with K whole, and on bf16 rows with a workspace."""
  got = []
  for rows, n in ((x.float(), 0), (x, 0), (x, ws_bytes)):
    out = torch.full(out_shape, float("nan"), dtype=dtype, device="cuda")
    ep, state = make(out)
    ws = torch.full((max(n, 16),), 0xFF, dtype=torch.uint8, device="cuda")
    lib.call("fh_gemm_bfp_ws", ops._ptr(rows), ops._TORCH[rows.dtype], rows.stride(0), rows.shape[0], bw.K, bw.N, ops._ptr(bw.mant),
             ops._ptr(bw.exps), lib.DTYPES[bw.fmt], ctypes.byref(ep) if ep is not None else None, ops._ptr(out), ops._TORCH[dtype],
             out.stride(0), ops._ptr(ws) if n else None, n, ops._stream())
    torch.cuda.synchronize()
    got.append([out, *state])
  return got


@pytest.mark.parametrize("fmt", ["bfp8", "bfp4"])
@pytest.mark.parametrize("M,K,N", list(PLANS))
def test_every_epilogue_at_tile_edges(cuda, fmt, M, K, N):
  from ferrite_amd import lib, ops
  g = torch.Generator(device="cuda").manual_seed(M + 3 * K + 7 * N)
  rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
  x = torch.full((M + 8, K), float("nan"), dtype=torch.bfloat16, device="cuda")
  x[:M] = rand(M, K)
  x = x[:M]
  n = parts_bytes(lib, M, K, N, PLANS[M, K, N])

  def check(bw, make, shape, dtype, bound, what):
    old, one, split = both(ops, lib, x, bw, make, shape, dtype, n)
    for a, b in zip(old, one): assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what
    for a, b in zip(old, split):
      if not n: assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what
      elif a.dtype in (torch.float32, torch.bfloat16): assert ((a.double() - b.double()).abs() <= bound(a.double())).all(), what

  w = rand(K, N) * 0.02
  bw = ops.pack(w, fmt)
  mag = (x.double().abs() @ ops.dequant(bw).double().abs())
  # sums of exact products in another order: K / 16 roundings a side, each of at most 2^-24 of a partial sum, which products of
  # random signs keep within 4 sum |x w| / sqrt(K); of random signs themselves, 2^-24 of sum |x w| in all whatever K, and
  # eight times that for the largest of millions of outputs
  near = 2 ** -21 * mag
  def store(out):
    parts = torch.zeros(M, N // 16, dtype=torch.int64, device="cuda")
    return ops.epilogue(lib.EP_STORE, argmax_parts=parts), [parts]
  check(bw, store, (M, N), torch.float32, lambda a: near, "store")
  # (bf16 on both sides: each rounding moves its sum by half a bf16 step, at most 2^-8 of it, so 2^-7 between the two)
  check(bw, lambda out: (None, []), (M, N), torch.bfloat16, lambda a: near + 2 ** -7 * a.abs(), "store bf16")
  res, cw = rand(M, N), rand(N)
  def residual(out):
    ssq, cp = torch.zeros(M, N // 16, device="cuda"), torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
    return ops.epilogue(lib.EP_RESIDUAL, residual=res, ssq_out=ssq, copy_bf16=cp, copy_w=cw), [ssq, cp]
  def residual_bound(a):
    if a.shape[1] != N: return 1e-4 * a + 1e-4  # the sums of squares: twice a value's error times the value, 16 of them
    return near * (1 + cw.abs()) + 2 ** -7 * a.abs()  # (the copy: two bf16 roundings, as above)
  check(bw, residual, (M, N), torch.float32, residual_bound, "residual")
  # 1/rms from the rows' own sums of squares
  ssq_in = x.float().square().reshape(M, K // 16, 16).sum(-1)
  check(bw, lambda out: (ops.epilogue(lib.EP_STORE, ssq_in=ssq_in, eps=1e-5), []), (M, N), torch.float32, lambda a: near, "1/rms")
  if N % 32 == 0:
    check(bw, lambda out: (ops.epilogue(lib.EP_SILU_GATE, split=N // 2), []), (M, N // 2), torch.bfloat16,
          lambda a: 2 ** -7 * a.abs() + 1e-5 * mag[:, :N // 2] * (1 + mag[:, N // 2:]), "silu")
  if N % (6 * HD) == 0:  # heads of 64: 4 of q's to each of k's and v's
    kv = N // (6 * HD)
    cos, sin = (torch.from_numpy(t).cuda() for t in G.rotary_tables(G.model(dim=HD, heads=1, theta=1e4), 64))
    places = torch.randint(0, 64, (M,), generator=g, device="cuda", dtype=torch.int32)
    rows = torch.randperm(M + 9, generator=g, device="cuda")[:M].to(torch.int32)
    for kind in ("fp32", "bfp8", "bfp4"):
      def rope(out):
        cache = ops.kv_cache(2 * kv, M + 9, HD, kind, "cuda")
        data, dt, length = ops.cache_fields(cache)
        ep = ops.epilogue(lib.EP_ROPE_KV, heads=4 * kv, kv_heads=kv, head_dim=HD, cos_tab=cos, sin_tab=sin, rope_rows=64, places=places,
                          cache_rows=rows, cache=data, cache_dtype=dt, cache_len=length)
        return ep, [data]
      big = 2 * near.max()
      check(bw, rope, (M, 4 * kv * HD), torch.float32, lambda a: big + 0 * a, f"rope {kind}")


def cache_parts(data, kind, rows):
  """A cache's values in 64 bits and the step its values lie on (a block float's run; 0 elsewhere), [rows][HD]."""
  if kind in ("fp32", "bf16"): return data.double().reshape(rows, HD), 0 * data.double().reshape(rows, HD)
  mags, e = data[:rows * HD // (1 if kind == "bfp8" else 2)], data[data.numel() - rows * HD // 16:].double()
  q, bias = (mags.view(torch.int8).double(), 133) if kind == "bfp8" else (torch.stack([mags.to(torch.int16) & 15, mags.to(torch.int16) >> 4], -1).double(), 129)
  if kind == "bfp4": q = torch.where(q > 7, q - 16, q)
  step = torch.exp2(e - bias)[:, None].expand(-1, 16)
  return (q.reshape(-1, 16) * step).reshape(rows, HD), step.reshape(rows, HD)


@pytest.mark.parametrize("kind", ["fp32", "bf16", "bfp8", "bfp4"])
@pytest.mark.parametrize("M,K,heads,kv", list(ROPES))
def test_rope_where_the_pairs_end_inside_a_tile(cuda, kind, M, K, heads, kv):
  """A qkv matmul whose pairs of runs are no whole tiles (SmolLM's 30 in tiles of 4 among them), rows at place 0 among
  the others, on fp32 rows, on bf16 rows with K whole (the same bits) and with K in parts (fp32 sums in another order; the
  cache's values each rounded to its format, so a step of each run's more)."""
  from ferrite_amd import lib, ops
  N = (heads + 2 * kv) * HD
  g = torch.Generator(device="cuda").manual_seed(M + K + heads)
  x = torch.full((M + 8, K), float("nan"), dtype=torch.bfloat16, device="cuda")
  x[:M] = torch.randn(M, K, generator=g, device="cuda")
  x = x[:M]
  bw = ops.pack(torch.randn(K, N, generator=g, device="cuda") * 0.02, "bfp8")
  cos, sin = (torch.from_numpy(t).cuda() for t in G.rotary_tables(G.model(dim=HD, heads=1, theta=1e4), 64))
  places = torch.arange(M, dtype=torch.int32, device="cuda") % 64
  rows = torch.randperm(M + 9, generator=g, device="cuda")[:M].to(torch.int32)
  def rope(out):
    cache = ops.kv_cache(2 * kv, M + 9, HD, kind, "cuda")
    data, dt, length = ops.cache_fields(cache)
    return ops.epilogue(lib.EP_ROPE_KV, heads=heads, kv_heads=kv, head_dim=HD, cos_tab=cos, sin_tab=sin, rope_rows=64, places=places,
                        cache_rows=rows, cache=data, cache_dtype=dt, cache_len=length), [data]
  old, one, split = both(ops, lib, x, bw, rope, (M, heads * HD), torch.float32, parts_bytes(lib, M, K, N, ROPES[M, K, heads, kv]))
  for a, b in zip(old, one): assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
  # against 64 bits: q turned by its row's place, k turned and v as they are in the cache rows
  y = (x.double() @ ops.dequant(bw).double()).reshape(M, -1, HD)
  turn = y[:, :heads + kv]
  c, s = cos[places].double()[:, None], sin[places].double()[:, None]
  y[:, :heads + kv] = turn * c + torch.cat([-turn[..., HD // 2:], turn[..., :HD // 2]], -1) * s
  # (sums of exact products in fp32, 2^-21 of sum |x w| as above, and a turn's two products and sum: of the two sums together)
  near = 4 * 2 ** -21 * (x.double().abs() @ ops.dequant(bw).double().abs()).max()
  for got in (one, split):
    assert ((got[0].double().reshape(M, heads, HD) - y[:, :heads]).abs() <= near).all()
    v, step = cache_parts(got[1], kind, 2 * kv * (M + 9))
    v, step = (t.reshape(2 * kv, M + 9, HD)[:, rows.long()].permute(1, 0, 2) for t in (v, step))
    want = y[:, heads:]
    # (bf16's rounding, then at most a whole step of a run's block float: the largest magnitudes saturate)
    assert ((v - want).abs() <= near + (0 if kind == "fp32" else 2 ** -8 * want.abs()) + step).all()
