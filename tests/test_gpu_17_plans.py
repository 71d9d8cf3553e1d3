"""Kernels at the sizes where a rule picks another plan for them, against plain float64 on the exact packed values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["bfp8", "bfp4"])
@pytest.mark.parametrize("rows", [1, 2, 8])
@pytest.mark.parametrize("K,N", [(1, 16), (63, 32), (64, 48), (65, 64), (576, 960), (1000, 576), (1536, 1536), (2048, 16), (4160, 4096), (4096, 4112)])
def test_gemv_slices(cuda, fmt, rows, K, N):
  """The GEMV's K slices: a wave as few as 64 rows where there are few items, as many as its loads in flight cover past
  that. Exact products summed in fp32: K roundings of at most 2^-24 of sum |x w| each, and far fewer in its tree."""
  from ferrite_amd import ops
  g = torch.Generator(device="cuda").manual_seed(K + 5 * N + rows)
  x = torch.randn(rows, K, generator=g, device="cuda")
  bw = ops.pack(torch.randn(K, N, generator=g, device="cuda") * 0.02, fmt)
  wv = ops.dequant(bw).double()
  got = ops.gemv(x, bw)
  assert ((got.double() - x.double() @ wv).abs() <= 2 ** -20 * (x.double().abs() @ wv.abs()) + 1e-30).all()


@pytest.mark.parametrize("kind", ["bf16", "fp32", "bfp8", "bfp4"])
@pytest.mark.parametrize("heads,kv,hd", [(4, 2, 128), (9, 3, 64)])
@pytest.mark.parametrize("T,p0", [(1, 0), (1, 64), (31, 33), (32, 64), (33, 63), (100, 0), (129, 100), (200, 824), (40, 1000)])
def test_prefill_attention_of_few_rows(cuda, kind, heads, kv, hd, T, p0):
  """A short prompt's causal attention, its keys split among a workgroup's waves (some of whose tiles lie wholly past a
  row), against float64 on the values the matrix cores take (bf16 q, k and v): the weights' bf16 rounding is at most 2^-9
  of each, and their sum's the same, so 2^-8 of the largest value. Cache rows past the prompt hold NaN."""
  from ferrite_amd import ops
  g = torch.Generator(device="cuda").manual_seed(T + 7 * p0 + heads)
  n = p0 + T
  q = torch.randn(T, heads * hd, generator=g, device="cuda")
  if kind in ("bf16", "fp32"):
    cache = torch.full((2 * kv, n + 70, hd), float("nan"), device="cuda", dtype=torch.bfloat16 if kind == "bf16" else torch.float32)
    cache[:, :n] = torch.randn(2 * kv, n, hd, generator=g, device="cuda")
    vals = cache[:, :n].to(torch.bfloat16).double()
  else:
    cache = ops.kv_cache(2 * kv, n + 70, hd, kind)
    rows = 2 * kv * (n + 70)
    mags = rows * hd // (1 if kind == "bfp8" else 2)
    m = torch.randint(-127, 128, (mags,), generator=g, device="cuda", dtype=torch.int16) if kind == "bfp8" else torch.randint(0, 256, (mags,), generator=g, device="cuda", dtype=torch.int16)
    if kind == "bfp4": m = torch.where((m & 15) == 8, m - 1, m); m = torch.where((m >> 4) == 8, m - 16, m)  # (no -8 in the format)
    cache.data[:mags] = m.to(torch.uint8)
    cache.data[mags:] = torch.randint(124, 128, (rows * hd // 16,), generator=g, device="cuda", dtype=torch.int16).to(torch.uint8)
    e = cache.data[mags:].double()
    if kind == "bfp8": v = cache.data[:mags].view(torch.int8).double()
    else:
      b = cache.data[:mags].to(torch.int16)
      v = torch.stack([b & 15, b >> 4], -1).reshape(-1)
      v = torch.where(v > 7, v - 16, v).double()
    vals = (v.reshape(-1, 16) * torch.exp2(e - (133 if kind == "bfp8" else 129))[:, None]).reshape(2 * kv, n + 70, hd)[:, :n]
  got = ops.attention_prefill(q, cache, heads, kv, hd, p0, 0).double().reshape(T, heads, hd)
  qb = q.to(torch.bfloat16).double().reshape(T, heads, hd)
  late = torch.arange(n, device="cuda")[None] > (p0 + torch.arange(T, device="cuda"))[:, None]
  for h in range(heads):
    k, v = vals[h // (heads // kv)], vals[kv + h // (heads // kv)]
    s = (qb[:, h] @ k.T.contiguous()) / hd ** 0.5
    want = torch.softmax(s.masked_fill(late, -torch.inf), -1) @ v
    assert ((got[:, h] - want).abs() <= 2 ** -8 * v.abs().max()).all(), h
