"""Matmul of plain operands (fh_matmul; Tensor.matmul with a bf16 or fp32 B, ferrite/tensor.py:443-485) against numpy,
after the reference's own checks (test/test_sim.py: test_matmul_exact 310-323, test_matmul_random 325-335,
test_matmul_blocks 337-354, test_fp32's fp32 matmul 870-880): small integers and x @ I bit for bit; x @ diag(d) with
full-mantissa d, each output one product, exact in fp32; random bf16 operands within a bf16 step of sum |a b| (bf16
out) or fp32 rounding of it (fp32 out); fp32 operands as bf16x3 within 2^-14 of sum |a b|, a bound bf16 operands
alone miss by far; batches and broadcasting; the elementwise chain on top fused into the same launch."""
import numpy as np
import pytest
import torch
from oracle import bfp as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt(cuda):
  from ferrite_amd import tensor
  return tensor.Runtime(0)


def Tn():
  from ferrite_amd import tensor
  return tensor.Tensor


def ops():
  from ferrite_amd import ops as o
  return o


def gpu(a, dtype):
  return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda").to(dtype)


def test_exact_integers_identity_and_diagonal(cuda):
  a = np.array([[float((r * 7 + c * 3) % 3 - 1) for c in range(64)] for r in range(32)], np.float32)
  b = np.array([[float((r * 5 + c) % 3 - 1) for c in range(32)] for r in range(64)], np.float32)
  want = a.astype(np.float64) @ b
  for da in (torch.bfloat16, torch.float32):
    for db in (torch.bfloat16, torch.float32):
      got = ops().matmul(gpu(a, da)[None], gpu(b, db)[None])[0].cpu().numpy()
      assert np.array_equal(got, want), (da, db)
  rng = np.random.default_rng(131)
  x = O.bf16(rng.uniform(-8, 8, (96, 64)))
  eye = np.eye(64, dtype=np.float32)
  assert np.array_equal(ops().matmul(gpu(x, torch.bfloat16)[None], gpu(eye, torch.bfloat16)[None])[0].cpu().numpy(), x)
  d = O.bf16(rng.uniform(1, 2, 64))
  got = ops().matmul(gpu(x, torch.bfloat16)[None], gpu(np.diag(d), torch.bfloat16)[None])[0].cpu().numpy()
  assert np.array_equal(got, (x.astype(np.float64) * d).astype(np.float32))  # one bf16 x bf16 product each: exact
  gb = ops().matmul(gpu(x, torch.bfloat16)[None], gpu(np.diag(d), torch.bfloat16)[None], out_dtype=torch.bfloat16)
  assert np.array_equal(gb[0].float().cpu().numpy(), O.bf16(x.astype(np.float64) * d))  # rounded once, to nearest even


def test_random_bf16_shapes(cuda):
  rng = np.random.default_rng(132)
  # (a 64 x 64 tile's edges: M, N and K not multiples of 64 or of the 32-k step; one row; one column of K)
  for M, K, N in ((64, 96, 128), (160, 96, 192), (1, 4096, 64), (45, 70, 33), (7, 1, 9), (130, 33, 65)):
    a, b = O.bf16(rng.uniform(-1, 1, (M, K))), O.bf16(rng.uniform(-1, 1, (K, N)))
    want = a.astype(np.float64) @ b
    mag = np.abs(a).astype(np.float64) @ np.abs(b)
    got = ops().matmul(gpu(a, torch.bfloat16)[None], gpu(b, torch.bfloat16)[None])[0].cpu().numpy()
    assert (np.abs(got - want) <= 2 ** -22 * mag + 1e-30).all(), (M, K, N)  # exact products, fp32 sums
    gb = ops().matmul(gpu(a, torch.bfloat16)[None], gpu(b, torch.bfloat16)[None], out_dtype=torch.bfloat16)[0].float().cpu().numpy()
    assert (np.abs(gb - want) <= 2 ** -8 * mag + 1e-30).all(), (M, K, N)


def test_fp32_operands_bf16x3(cuda):
  rng = np.random.default_rng(133)
  for M, K, N in ((45, 70, 33), (128, 512, 96)):
    a, b = rng.uniform(-2, 2, (M, K)).astype(np.float32), rng.uniform(-2, 2, (K, N)).astype(np.float32)
    want = a.astype(np.float64) @ b
    mag = np.abs(a).astype(np.float64) @ np.abs(b)
    got = ops().matmul(gpu(a, torch.float32)[None], gpu(b, torch.float32)[None])[0].cpu().numpy()
    err = np.abs(got - want) / mag
    assert err.max() <= 2 ** -14, err.max()
    # bf16 operands alone are far off that bound: the lo parts are in the sum
    bf = ops().matmul(gpu(a, torch.bfloat16)[None], gpu(b, torch.bfloat16)[None])[0].cpu().numpy()
    assert (np.abs(bf - want) / mag).max() > 2 ** -12
    # one fp32 operand: its lo part with the other's hi (hi@hi + hi@lo or lo@hi)
    ab = O.bf16(a)
    got = ops().matmul(gpu(ab, torch.bfloat16)[None], gpu(b, torch.float32)[None])[0].cpu().numpy()
    assert (np.abs(got - ab.astype(np.float64) @ b) / mag).max() <= 2 ** -14


def test_batches_and_broadcast(cuda):
  rng = np.random.default_rng(134)
  a3, b3 = O.bf16(rng.normal(0, 1, (3, 20, 48))), O.bf16(rng.normal(0, 1, (3, 48, 40)))
  a1, b1 = a3[:1], b3[:1]
  for a, b in ((a3, b3), (a3, b1), (a1, b3)):
    want = np.einsum("bmk,bkn->bmn", np.broadcast_to(a, (3,) + a.shape[1:]).astype(np.float64), np.broadcast_to(b, (3,) + b.shape[1:]))
    got = ops().matmul(gpu(a, torch.bfloat16), gpu(b, torch.bfloat16)).cpu().numpy()
    assert got.shape == (3, 20, 40)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()


def test_rejects(cuda):
  a = torch.zeros(1, 4, 8, device="cuda", dtype=torch.bfloat16)
  with pytest.raises(ValueError): ops().matmul(a, torch.zeros(1, 9, 4, device="cuda", dtype=torch.bfloat16))
  with pytest.raises(ValueError): ops().matmul(a, torch.zeros(1, 8, 4, device="cuda", dtype=torch.int32))
  with pytest.raises(ValueError): ops().matmul(torch.zeros(2, 4, 8, device="cuda"), torch.zeros(3, 8, 4, device="cuda"))


def test_tensor_matmul_plain_with_its_chain(rt):
  rng = np.random.default_rng(135)
  x, w = O.bf16(rng.normal(0, 1, (37, 80))), O.bf16(rng.normal(0, 0.1, (80, 50)))
  bias = O.bf16(rng.normal(0, 1, (1, 50)))
  X, W, Bv = Tn().of(rt, x.tolist()), Tn().of(rt, w.tolist()), Tn().of(rt, bias.tolist())
  y = (X @ W + Bv).relu() * 0.5
  assert y.dtype == "bf16"
  before = rt.launches
  got = np.array(y.tolist(), np.float64)
  assert rt.launches - before == 1, rt.launches - before  # the matmul and its chain: one launch
  want = np.maximum(x.astype(np.float64) @ w + bias, 0) * 0.5
  assert (np.abs(got - O.bf16(want)) <= 2 ** -8 * np.abs(want) + 2 ** -8 * (np.abs(x) @ np.abs(w)) * 2 ** -7 + 1e-6).all()
  # fp32 operands, a batch by one matrix, the result fp32 (ferrite's dtype rule), and a transposed operand's view
  a = rng.uniform(-1, 1, (2, 9, 30)).astype(np.float32)
  A, Wt = Tn().of(rt, a.tolist(), "fp32"), Tn().of(rt, w[:30, :20].T.tolist(), "fp32")
  z = A @ Wt.T
  assert z.dtype == "fp32" and z.shape == (2, 9, 20)
  want = a.astype(np.float64) @ w[:30, :20]
  assert np.abs(np.array(z.tolist()) - want).max() <= 2 ** -14 * (np.abs(a) @ np.abs(w[:30, :20])).max()


@pytest.mark.parametrize("M,K,N", [
  (1, 64, 8), (129, 64, 136), (255, 128, 264),      # a tile and a row or a piece more or less; one K step, two
  (2047, 192, 2048), (2049, 256, 2056),             # 128 x 128 tiles from LDS loads: 3 and 4 steps of a 4-stage ring
  (4095, 320, 4104),                                # 128 x 256 tiles, 5 steps of a 3-stage ring
  (2048, 66, 2050), (4097, 130, 4099),              # K past whole steps, odd rows: 128 and 256 wide tiles by registers
  (300, 60, 1001),
])
def test_tiles_and_strides_give_the_same_bits(cuda, M, K, N):
  """Each kernel and tile against the sums in float64 (exact products, fp32 sums over at most K / 16 chained MFMAs:
  2^-21 of sum |a b|), and operands at odd and at even strides against the contiguous ones, bit for bit (the products
  come in one order in every kernel). Rows and columns past M and N hold NaN: none of them may reach a sum."""
  g = torch.Generator(device="cuda").manual_seed(M * 7 + K * 3 + N)
  a, b = (torch.randn(1, *s, generator=g, device="cuda").to(torch.bfloat16) for s in ((M, K), (K, N)))
  got = ops().matmul(a, b)
  want, mag = a.double()[0] @ b.double()[0], a.double()[0].abs() @ b.double()[0].abs()
  assert ((got[0].double() - want).abs() <= 2 ** -21 * mag).all()
  for pad in (1, 2, 8):
    wide = [torch.full((1, t.shape[1], t.shape[2] + pad), float("nan"), dtype=t.dtype, device="cuda") for t in (a, b)]
    for w, t in zip(wide, (a, b)): w[:, :, :t.shape[2]] = t
    again = ops().matmul(wide[0][:, :, :K], wide[1][:, :, :N])
    assert torch.equal(again, got), pad
  half = ops().matmul(a, b, out_dtype=torch.bfloat16)
  assert torch.equal(half, got.to(torch.bfloat16))  # rounded once, to nearest even, in vector and in single stores


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16, torch.int32])
@pytest.mark.parametrize("batch,M,K,N", [
  (3, 5, 33, 17), (1, 64, 64, 64), (2, 65, 64, 63),   # 64 x 64 tiles: inside one, one whole, a row more and a column less
  (1, 2047, 64, 2056),                                # 128 x 128 from LDS loads, the last row and piece past whole tiles
  (1, 4095, 64, 4104), (1, 4097, 16, 4099),           # 128 x 256 from LDS loads; 256 x 256 by registers
])
def test_programs_give_the_elementwise_kernels_bits(cuda, batch, M, K, N, out_dtype):
  """A matmul's program against the plain matmul followed by the same program in the elementwise kernel, bit for bit:
  15 ops, every op in one of the three programs, operands from results far back, immediates, the matmul's result and
  inputs of each type (one broadcast over rows, one over columns), at the tiles' edges and for fp32 operands too; C's
  places between its rows stay as they were."""
  import ctypes
  from ferrite_amd import lib
  g = torch.Generator(device="cuda").manual_seed(batch + M + K + N)
  rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
  ins = [rnd(batch, M, N), rnd(batch, 1, N).to(torch.bfloat16), torch.randint(-9, 9, (1, M, 1), generator=g, device="cuda", dtype=torch.int32)]
  strides = [(M * N, N, 1), (N, 0, 1), (0, 1, 0)]
  acc, imm, x, y, z = lib.OPND_ACC, lib.OPND_IMM, 16, 17, 18
  programs = [
    [("add", acc, x), ("mul", 0, y), ("sub", 1, z), ("max", 2, acc), ("cmplt", 0, 3), ("cmpne", 1, imm, 0.5), ("keep", 4, 2), ("drop", 4, x),
     ("add", 6, 7), ("relu", 8, 8), ("sin", 0, 0), ("cos", 10, 10), ("mul", 9, 11), ("add", 12, 5), ("sub", 13, 0)],
    [("relu", acc, acc), ("add", 0, imm, 1.0), ("log", 1, 1), ("log2", 1, 1), ("sqrt", 1, 1), ("recip", 4, 4), ("exp", 5, 5), ("exp2", 2, 2),
     ("add", 6, 7), ("mul", 8, 3), ("ftob", 9, 9), ("max", 10, y), ("itof", z, z), ("add", 11, 12), ("copy", 13, 13)],
    [("ftoi", acc, acc)]]
  def made(ops_, inputs, st):
    p = lib.Program()
    p.n_ops, p.n_inputs = len(ops_), len(inputs)
    for k, (t, s) in enumerate(zip(inputs, st)):
      p.input[k], p.in_dtype[k] = t.data_ptr(), {torch.float32: lib.F32, torch.bfloat16: lib.BF16, torch.int32: lib.I32}[t.dtype]
      for i in range(3): p.in_stride[k][i] = s[i]
    for i, o in enumerate(ops_): p.op[i], p.a[i], p.b[i], p.imm[i] = lib.OP[o[0]], o[1], o[2], o[3] if len(o) > 3 else 0.0
    return p
  out_code = {torch.float32: lib.F32, torch.bfloat16: lib.BF16, torch.int32: lib.I32}[out_dtype]
  a, b = rnd(batch, M, K), rnd(batch, K, N)
  for da, db in ((torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)):
    A, B = a.to(da), b.to(db)
    plain = ops().matmul(A, B)
    for prog in programs:
      swap = [tuple(19 if i in (1, 2) and v == acc else v for i, v in enumerate(o)) for o in prog]
      q = made(swap, ins + [plain], strides + [(M * N, N, 1)])
      want = torch.empty(batch, M, N, device="cuda", dtype=out_dtype)
      lib.call("fh_map", ctypes.byref(q), want.data_ptr(), out_code, batch, M, N, M * N, N, ops()._stream())
      for pad in (0, 3):
        wide = torch.full((batch, M, N + pad), 77, device="cuda", dtype=out_dtype)
        ops().matmul(A, B, made(prog, ins, strides), out=wide[:, :, :N])
        assert torch.equal(wide[:, :, :N], want), (da, len(prog), pad)
        assert (wide[:, :, N:] == 77).all()
