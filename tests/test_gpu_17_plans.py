"""Kernels at the sizes where a rule picks another plan for them, against plain float64 on the exact packed values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["bfp8", "bfp4"])
@pytest.mark.parametrize("rows", [1, 2, 8])
@pytest.mark.parametrize("K,N", [(1, 16), (63, 32), (64, 48), (65, 64), (576, 960), (1000, 576), (1536, 1536), (2048, 16), (4160, 4096), (4096, 4112)])
def test_gemv_slices(cuda, fmt, rows, K, N):
  """The GEMV's K slices: whole groups of a wave's loads in flight, the last a part of one, at edges of 64 rows and of the
  groups. Exact products summed in fp32: K roundings of at most 2^-24 of sum |x w| each, and far fewer in its tree."""
  from ferrite_amd import ops
  g = torch.Generator(device="cuda").manual_seed(K + 5 * N + rows)
  x = torch.randn(rows, K, generator=g, device="cuda")
  bw = ops.pack(torch.randn(K, N, generator=g, device="cuda") * 0.02, fmt)
  wv = ops.dequant(bw).double()
  got = ops.gemv(x, bw)
  assert ((got.double() - x.double() @ wv).abs() <= 2 ** -20 * (x.double().abs() @ wv.abs()) + 1e-30).all()


@pytest.mark.parametrize("kind", ["bf16", "fp32", "bfp8", "bfp4"])
@pytest.mark.parametrize("heads,kv,hd", [(4, 2, 128), (9, 3, 64)])
@pytest.mark.parametrize("T,p0", [(1, 0), (1, 64), (31, 33), (32, 64), (33, 63), (100, 0), (129, 100), (200, 824), (40, 1000),
                                  (1, 320), (33, 320), (60, 300)])
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


@pytest.mark.parametrize("fmt", ["bfp8", "bfp4"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N,pad,off", [(16, 16, 0, 0), (63, 272, 0, 0), (64, 256, 8, 0), (65, 240, 4, 0), (128, 4112, 0, 0), (80, 64, 1, 0), (96, 48, 0, 1),
                                         (2064, 1040, 0, 0), (1, 2097152, 0, 0), (7, 299600, 0, 0), (8, 262160, 8, 0), (9, 240000, 2, 0), (1104, 2064, 2, 0), (2048, 1072, 8, 1), (4096, 4112, 0, 0), (4112, 4104, 4, 0)])
def test_packing_at_every_stride(cuda, fmt, dtype, K, N, pad, off):
  """fh_bfp_pack along both axes, in its wide and its narrow loads (whole tiles and ragged ones, row strides and bases at
  odd alignments), against the oracle's blocks: magnitudes and exponents bit for bit, as gpt2.bfp makes them."""
  import numpy as np
  from ferrite_amd import lib, ops
  from oracle import bfp as O
  rng = np.random.default_rng(K + N + pad)
  w = (rng.normal(0, 1, (K, N)) * np.exp(rng.normal(0, 3, (K, N)))).astype(np.float32)
  w[rng.random((K, N)) < 0.05] = 0
  buf = torch.full((off + K * (N + pad),), float("nan"), dtype=dtype, device="cuda")
  x = buf[off:].view(K, N + pad)[:, :N]
  x.copy_(torch.from_numpy(w))
  vals = x.float().cpu().numpy()
  for axis in (lib.AXIS_N, lib.AXIS_K):
    if (K if axis == lib.AXIS_K else N) % 16: continue
    bw = ops.pack(x, fmt, axis)
    q, top = O.bfp_parts(vals if axis == lib.AXIS_N else vals.T, fmt)  # [inner][outer * 16], [inner][outer]
    assert np.array_equal(bw.exps.cpu().numpy().reshape(top.shape[1], top.shape[0]), top.T), axis
    m = bw.mant.cpu().numpy().reshape(top.shape[1], top.shape[0], -1)
    if fmt == "bfp8": got = m.view(np.int8).astype(np.int32)
    else:
      got = np.stack([m & 15, m >> 4], -1).reshape(*m.shape[:2], 16).astype(np.int32)
      got = np.where(got > 7, got - 16, got)
    assert np.array_equal(got, q.reshape(q.shape[0], -1, 16).transpose(1, 0, 2)), axis


@pytest.mark.parametrize("M,K,N", [(200, 64, 33600), (200, 96, 51200), (300, 64, 51200), (65, 96, 640), (2048, 96, 6144)])
def test_gemm_program_tiles(cuda, M, K, N):
  """A fused elementwise program on bf16 rows' matmul (the kernels that fh_gemm_lds.hip's does not replace: programs, and a
  K that is not whole steps of 64), in each of their tile widths, against float64: exact products, fp32 sums."""
  import ctypes
  from ferrite_amd import lib, ops
  g = torch.Generator(device="cuda").manual_seed(M + N)
  x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
  bw = ops.pack(torch.randn(K, N, generator=g, device="cuda") * 0.02, "bfp8")
  wv = ops.dequant(bw).double()
  mag, want = x.double().abs() @ wv.abs(), x.double() @ wv
  p = lib.Program()
  p.n_ops, p.op[0], p.a[0], p.b[0], p.imm[0] = 1, lib.OP["mul"], lib.OPND_ACC, lib.OPND_IMM, 0.5
  for program, scale in ((p, 0.5), (None, 1.0)):
    ep = ops.epilogue(lib.EP_PROGRAM if program is not None else lib.EP_STORE)
    if program is not None: ep.program = ctypes.pointer(program)
    got = ops.gemm(x, bw, ep)
    assert ((got.double() - scale * want).abs() <= 2 ** -21 * mag + 1e-30).all()


@pytest.mark.parametrize("M", [33, 36, 47, 48, 49])
@pytest.mark.parametrize("K,N", [(64, 48), (576, 960), (1536, 576)])
def test_tile_rows_between_block_counts(cuda, M, K, N):
  """Rows in tiles of 16 where the kernel's blocks (4) are more than the rows' tiles (3 for 33 to 48 rows): the tiles past
  the last are not read (the buffer ends there), and the outputs are the plain rows', bit for bit."""
  from ferrite_amd import ops
  g = torch.Generator(device="cuda").manual_seed(M + K)
  x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
  bw = ops.pack(torch.randn(K, N, generator=g, device="cuda") * 0.02, "bfp8")
  assert torch.equal(ops.gemm(ops.to_tiles16(x, float("nan")), bw), ops.gemm(x, bw))


@pytest.mark.parametrize("rows,sized", [(512, 513), (512, 600), (300, 513), (129, 257)])
def test_moe_in_a_workspace_sized_for_more_rows(cuda, rows, sized):
  """down's K goes in parts for 65 to 512 rows only, so more rows' workspace can be the smaller one: it still serves fewer
  rows (in the parts that fit), with the larger workspace's results but for the order of fp32 sums of its 4096 products."""
  from ferrite_amd import lib, ops
  E, dim, ffn = 2, 256, 4096
  g = torch.Generator(device="cuda").manual_seed(rows)
  gu, dn = (torch.randn(*s, generator=g, device="cuda") * 0.05 for s in ((E, dim, 2 * ffn), (E, ffn, dim)))
  ex = ops.pack_experts(gu, dn, "bfp8")
  x = torch.randn(rows, dim, generator=g, device="cuda")
  dense = torch.rand(rows, E, generator=g, device="cuda")
  want = ops.moe_experts(x, ex, dense)
  need, have = lib.load().fh_moe_workspace_bytes(rows, E, ffn, dim), lib.load().fh_moe_workspace_bytes(sized, E, ffn, dim)
  ws, got = torch.empty(have, dtype=torch.uint8, device="cuda"), torch.empty(rows, dim, device="cuda")
  lib.call("fh_moe_experts", x.data_ptr(), dim, rows, dim, None, None, 1e-5, 0, E, ffn, ex.gate_up.mant.data_ptr(), ex.gate_up.exps.data_ptr(),
           lib.DTYPES["bfp8"], ex.down.mant.data_ptr(), ex.down.exps.data_ptr(), lib.DTYPES["bfp8"], dense.data_ptr(), got.data_ptr(),
           None, None, ws.data_ptr(), have, torch.cuda.current_stream().cuda_stream)
  if sized == 513 and rows == 512: assert need > have
  # (4096 products an expert summed in fp32 in 16s on the matrix cores: fewer than 2^9 roundings of 2^-24 of the sum of
  # their magnitudes in each order; twice that sum as plain fp32 has it covers the rounding of h and the weights)
  mag = sum(dense[:, e:e + 1] * ((torch.nn.functional.silu(x @ gu[e, :, :ffn]) * (x @ gu[e, :, ffn:])).abs() @ dn[e].abs()) for e in range(E))
  assert ((got - want).abs() <= 2 * 2 * 2 ** -15 * mag).all()


@pytest.mark.parametrize("rows", [65, 300, 512, 513])
def test_moe_in_a_workspace_at_8_bytes(cuda, rows):
  """A workspace that is not 16-byte aligned serves too: down's K whole there, whatever the rows (fh_gemm_lds.hip, which
  takes K in parts, reads 16-byte aligned rows), the results as in an aligned one but for the order of fp32 sums."""
  from ferrite_amd import lib, ops
  E, dim, ffn = 2, 256, 2048
  g = torch.Generator(device="cuda").manual_seed(rows)
  gu, dn = (torch.randn(*s, generator=g, device="cuda") * 0.05 for s in ((E, dim, 2 * ffn), (E, ffn, dim)))
  ex = ops.pack_experts(gu, dn, "bfp4")
  x = torch.randn(rows, dim, generator=g, device="cuda")
  dense = torch.rand(rows, E, generator=g, device="cuda")
  need = lib.load().fh_moe_workspace_bytes(rows, E, ffn, dim)
  want = ops.moe_experts(x, ex, dense, ws=torch.empty(need, dtype=torch.uint8, device="cuda"))
  ws = torch.full((need + 16,), 0xFF, dtype=torch.uint8, device="cuda")[8:]
  assert ws.data_ptr() % 16 == 8
  got = ops.moe_experts(x, ex, dense, ws=ws)
  # (2048 products an expert summed in fp32 16 at a time: fewer than 2^8 roundings of 2^-24 of the sum of their magnitudes
  # in each order; twice that sum, as above)
  mag = sum(dense[:, e:e + 1] * ((torch.nn.functional.silu(x @ gu[e, :, :ffn]) * (x @ gu[e, :, ffn:])).abs() @ dn[e].abs()) for e in range(E))
  assert ((got - want).abs() <= 2 * 2 * 2 ** -16 * mag).all()


def test_gemm_workspace_only_where_a_kernel_reads_it(cuda):
  """ops.gemm takes memory for K's parts only for the calls whose kernel adds them: a fused program, a norm's weight and
  rows off 16 bytes go to kernels that take K whole. A plain call takes the parts' bytes."""
  import ctypes
  from ferrite_amd import lib, ops
  M, K, N = 200, 4096, 1024
  g = torch.Generator(device="cuda").manual_seed(3)
  rows = torch.randn(M, K + 8, generator=g, device="cuda").to(torch.bfloat16)
  x, off = rows[:, :K], rows.view(-1)[4:4 + (M - 1) * (K + 8) + K].as_strided((M, K), (K + 8, 1))
  bw = ops.pack(torch.randn(K, N, generator=g, device="cuda") * 0.02, "bfp8")
  parts = lib.load().fh_gemm_workspace_bytes(M, K, N)
  out = torch.empty(M, N, device="cuda")
  assert parts > 1 << 20
  def program(op):
    p = lib.Program()
    p.n_ops, p.op[0], p.a[0], p.b[0], p.imm[0] = 1, lib.OP[op], lib.OPND_ACC, lib.OPND_IMM, 0.5
    ep = ops.epilogue(lib.EP_PROGRAM)
    ep.program = ctypes.pointer(p)
    return ep
  ssq, w = x.float().square().reshape(M, K // 16, 16).sum(-1), torch.ones(K, device="cuda")
  for rows_, ep, most in ((x, None, parts), (x, ops.epilogue(lib.EP_STORE, ssq_in=ssq, eps=1e-5), parts), (x, program("copy"), parts),
                          (x, program("mul"), 0), (x, ops.epilogue(lib.EP_STORE, norm_w=w, ssq_in=ssq, eps=1e-5), 0), (off, None, 0)):
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.gemm(rows_, bw, ep, out=out)
    took = torch.cuda.max_memory_allocated() - before
    assert took >= parts if most else took == 0, (took, most)


def test_gemm_without_room_for_its_parts(cuda, monkeypatch):
  """A card too full for K's parts: K whole, the bits of fh_gemm_bfp, which needs no workspace."""
  from ferrite_amd import lib, ops
  M, K, N = 200, 4096, 1024
  g = torch.Generator(device="cuda").manual_seed(4)
  x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
  bw = ops.pack(torch.randn(K, N, generator=g, device="cuda") * 0.02, "bfp4")
  want = torch.empty(M, N, device="cuda")
  lib.call("fh_gemm_bfp", x.data_ptr(), lib.BF16, K, M, K, N, bw.mant.data_ptr(), bw.exps.data_ptr(), lib.BFP4, None, want.data_ptr(),
           lib.F32, N, torch.cuda.current_stream().cuda_stream)
  monkeypatch.setattr(ops, "_gemm_workspace_bytes", lambda *a: 1 << 46)
  assert torch.equal(ops.gemm(x, bw), want)


def test_moe_experts_keeps_a_workspace_for_more_rows(cuda):
  """ops.moe_experts runs in the workspace it is given where that is one for more rows than the call's, though fewer rows'
  own, with its parts of down's K, would be larger; one for fewer rows it replaces."""
  from ferrite_amd import lib, ops
  E, dim, ffn = 2, 256, 4096
  g = torch.Generator(device="cuda").manual_seed(5)
  ex = ops.pack_experts(*(torch.randn(*s, generator=g, device="cuda") * 0.05 for s in ((E, dim, 2 * ffn), (E, ffn, dim))), "bfp8")
  bytes_ = lambda rows: lib.load().fh_moe_workspace_bytes(rows, E, ffn, dim)
  assert bytes_(512) > bytes_(513)
  for rows, sized, more in ((512, 513, False), (65, 513, False), (512, 2048, False), (512, 512, False), (512, 65, True), (600, 513, True)):
    x, dense, out = torch.randn(rows, dim, generator=g, device="cuda"), torch.rand(rows, E, generator=g, device="cuda"), torch.empty(rows, dim, device="cuda")
    ws = torch.empty(bytes_(sized), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.moe_experts(x, ex, dense, out=out, ws=ws)
    assert (torch.cuda.max_memory_allocated() > before) == more, (rows, sized)


@pytest.mark.parametrize("kind", ["fp32", "bf16", "norm"])
@pytest.mark.parametrize("M,K,N", [(65, 96, 48), (129, 96, 272), (300, 64, 640), (2048, 64, 1552), (1700, 128, 6144), (2048, 64, 8208)])
def test_gemm_programs_give_the_elementwise_kernels_bits(cuda, kind, M, K, N):
  """A block-float matmul's program past 64 rows (128 and 256 row tiles, the two-group kernel's widths; rows and runs past the
  matrix in the last tiles) against the plain store of the same kernels followed by the same program in the elementwise
  kernel, bit for bit: fp32 and bf16 outputs, inputs by row, by column and by both."""
  import ctypes
  from ferrite_amd import lib, ops
  g = torch.Generator(device="cuda").manual_seed(M + K + N)
  rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
  x = rnd(M, K) if kind != "bf16" else rnd(M, K).to(torch.bfloat16)
  bw = ops.pack(rnd(K, N) * 0.1, "bfp4" if M % 2 else "bfp8")
  norm = {"norm_w": rnd(K), "ssq_in": x.float().square().reshape(M, K // 16, 16).sum(-1), "eps": 1e-5} if kind == "norm" else {}
  ins, strides = [rnd(M, N), rnd(N).to(torch.bfloat16), rnd(M)], [(0, N, 1), (0, 0, 1), (0, 1, 0)]
  chain = [("mul", lib.OPND_ACC, 17), ("add", 0, 16), ("sub", 1, 18), ("exp2", 0, 0), ("max", 2, lib.OPND_ACC), ("cmplt", 3, 4), ("keep", 5, 2), ("add", 6, 1)]
  def made(ops_, inputs, st):
    p = lib.Program()
    p.n_ops, p.n_inputs = len(ops_), len(inputs)
    for k, (t, s) in enumerate(zip(inputs, st)):
      p.input[k], p.in_dtype[k] = t.data_ptr(), lib.BF16 if t.dtype == torch.bfloat16 else lib.F32
      for i in range(3): p.in_stride[k][i] = s[i]
    for i, (op, a, b) in enumerate(ops_): p.op[i], p.a[i], p.b[i] = lib.OP[op], a, b
    return p
  # (the plain sums by the same kernels: a program that gives them back)
  plain = ops.epilogue(lib.EP_PROGRAM, **norm)
  plain.program = ctypes.pointer(made([("copy", lib.OPND_ACC, lib.OPND_ACC), ("copy", 0, 0)], [], []))
  sums = ops.gemm(x, bw, plain)
  w = ops.dequant(bw).double()
  xs = x.double() if kind != "norm" else x.double() * norm["norm_w"].double() / (x.double().square().mean(-1, keepdim=True) + 1e-5).sqrt()
  assert ((sums.double() - xs @ w).abs() <= 2 ** -7 * (xs.abs() @ w.abs())).all()  # (rows rounded to bf16 for the matrix cores)
  ep = ops.epilogue(lib.EP_PROGRAM, **norm)
  ep.program = ctypes.pointer(made(chain, ins, strides))
  swapped = made([(op, *(19 if v == lib.OPND_ACC else v for v in ab)) for op, *ab in chain], ins + [sums], strides + [(0, N, 1)])
  for dt, code in ((torch.float32, lib.F32), (torch.bfloat16, lib.BF16)):
    want = torch.empty(M, N, device="cuda", dtype=dt)
    lib.call("fh_map", ctypes.byref(swapped), want.data_ptr(), code, 1, M, N, M * N, N, ops._stream())
    wide = torch.full((M, N + 8), 77, device="cuda", dtype=dt)
    ops.gemm(x, bw, ep, out=wide[:, :N])
    assert torch.equal(wide[:, :N], want), dt
    assert (wide[:, N:] == 77).all()
