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
