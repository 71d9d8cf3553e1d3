"""The work this framework does for a program that uses it, as cases that can be timed and checked: single matmuls by a
block float, decode steps and prompts of a Llama-shape model, decode attention over long contexts, a mixture of experts'
layer, the lazy Tensor's matmul, and packing weights. listed() names the cases, draw() gives more of the same ranges,
prepare() makes what a program holds before the call, run() is one pass through the public entry points, and exact()
the same outputs in 64 bits by plain torch."""
import math
import numpy as np
import torch
from ferrite_amd import llama, ops
from ferrite_amd.tensor import Runtime, Tensor

DEV = "cuda"

# Model shapes: SmolLM-135M (config 2 of the benchmark), Llama-3.1-8B (configs 3 and 4; a few of its 32 blocks, with the
# whole output layer) and a generic one between them.
MODELS = {
  "smollm-135m": dict(dim=576, heads=9, kv=3, eps=1e-5, theta=10000.0, vocab=49152, ffn=1536, tied=True),
  "llama-8b": dict(dim=4096, heads=32, kv=8, eps=1e-5, theta=500000.0, vocab=128256, ffn=14336, tied=False),
  "generic-2k": dict(dim=2048, heads=32, kv=8, eps=1e-5, theta=10000.0, vocab=32000, ffn=5632, tied=False),
}
LAYERS = {"smollm-135m": 30, "llama-8b": 4, "generic-2k": 8}
# Attention's heads, key heads and head_dim in those models, and the mixture's widths (config 5's Mixtral shape, and a
# generic one): dim, ffn.
HEADS = {"smollm-135m": (9, 3, 64), "llama-8b": (32, 8, 128), "generic-2k": (32, 8, 64)}
MOE = {"mixtral": (4096, 14336), "generic-2k": (2048, 5632)}
EXPERTS, TOP = 8, 2


def listed():
  return [
    # the smallest call: one token's row by one SmolLM matrix (the benchmark's config 1)
    dict(name="matmul 1x576x1536 bfp8", kind="matmul", rows=1, K=576, N=1536, fmt="bfp8", x="fp32"),
    # a batched service's projection called by itself: 24 rows by an 8B-shape o matrix
    dict(name="matmul 24x4096x4096 bfp8", kind="matmul", rows=24, K=4096, N=4096, fmt="bfp8", x="bf16"),
    # one user's next token on a small model: the whole 30-block SmolLM step (config 2)
    dict(name="decode smollm b1", kind="decode", model="smollm-135m", layers=30, mode="bfp8", kv="bf16", batch=1, cache=256, place=143),
    # one user's next token on an 8B-shape model at context 2048 (config 3), four of its blocks and the output layer
    dict(name="decode 8b b1", kind="decode", model="llama-8b", layers=4, mode="experts", kv="bf16", batch=1, cache=2048, place=2047),
    # a service's batch of 16 users at contexts of 1024 to 2048 (config 3's batch 16)
    dict(name="decode 8b b16", kind="decode", model="llama-8b", layers=4, mode="experts", kv="bf16", batch=16, cache=2048, place=2047),
    # a long prompt (config 4), two blocks and the last token's output layer
    dict(name="prefill 8b 2048", kind="prefill", model="llama-8b", layers=2, mode="bfp8", kv="bf16", tokens=2048, p0=0),
    # a chat turn of ordinary length, its 200 tokens after 824 cached ones
    dict(name="prefill 8b 200 of 1024", kind="prefill", model="llama-8b", layers=4, mode="experts", kv="bf16", tokens=200, p0=824),
    # decode attention by itself over long contexts
    dict(name="attend 8b b4 32k", kind="attend", model="llama-8b", kv="bf16", batch=4, context=32768),
    # a mixture's layer for a decode step of 32 users (config 5) and for a prompt of 300 tokens
    dict(name="moe mixtral 32", kind="moe", model="mixtral", rows=32, fmt="bfp4"),
    dict(name="moe mixtral 300", kind="moe", model="mixtral", rows=300, fmt="bfp4"),
    # the lazy Tensor's plain matmul at the size of the reference's own matmul benchmark (4096^3 in bf16)
    dict(name="tensor 4096^3 bf16", kind="tensor", M=4096, K=4096, N=4096, a="bf16", b="bf16"),
    # a model's upload: an 8B-shape block's gate and up matrices packed from a checkpoint's rows
    dict(name="pack 8b gate_up bfp4", kind="pack", K=4096, parts=2, out=14336, dtype="bf16", fmt="bfp4"),
  ]


def _log(rng, lo, hi, step=1):
  """A multiple of step between lo and hi, spread over their logarithm."""
  return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step) * step))


def draw(rng):
  kind = rng.choice(["matmul", "decode", "prefill", "attend", "moe", "tensor", "pack"])
  model = rng.choice(list(MODELS))
  if kind == "matmul":
    return dict(kind=kind, rows=_log(rng, 1, 1024), K=_log(rng, 256, 14336, 64), N=_log(rng, 256, 28672, 16),
                fmt=rng.choice(["bfp8", "bfp4"]), x=rng.choice(["fp32", "bf16"]))
  if kind == "decode":
    cache = _log(rng, 64, 4096, 8)
    return dict(kind=kind, model=model, layers=LAYERS[model], mode=rng.choice(["bfp8", "bfp4", "experts"]),
                kv=rng.choice(["bf16", "fp32", "bfp8", "bfp4"]), batch=_log(rng, 1, 64), cache=cache,
                place=rng.randrange(cache // 2, cache))
  if kind == "prefill":
    tokens = _log(rng, 8, 2048)
    return dict(kind=kind, model=model, layers=2 if model == "llama-8b" else LAYERS[model], mode=rng.choice(["bfp8", "bfp4", "experts"]),
                kv=rng.choice(["bf16", "bfp8"]), tokens=tokens, p0=rng.choice([0, 0, rng.randrange(1, 2049 - min(tokens, 2047))]))
  if kind == "attend":
    batch = _log(rng, 1, 16)
    return dict(kind=kind, model=model, kv=rng.choice(["bf16", "fp32", "bfp8", "bfp4"]), batch=batch,
                context=_log(rng, 1024, 131072 // max(batch, 2)))
  if kind == "moe":
    return dict(kind=kind, model=rng.choice(list(MOE)), rows=_log(rng, 1, 300), fmt=rng.choice(["bfp8", "bfp4", "bfp4"]))
  if kind == "tensor":
    a = rng.choice(["bf16", "bf16", "fp32"])
    top = 4096 if a == "bf16" else 2048
    return dict(kind=kind, M=_log(rng, 32, top), K=_log(rng, 64, top, 4), N=_log(rng, 32, top, 4), a=a, b=a)
  return dict(kind=kind, K=_log(rng, 512, 8192, 16), parts=rng.choice([0, 1, 2, 3]), out=_log(rng, 256, 8192, 16),
              dtype=rng.choice(["bf16", "fp32"]), fmt=rng.choice(["bfp8", "bfp4"]))


# ---- inputs ----------------------------------------------------------------------------------------------------------
def _gen(seed, name):
  g = torch.Generator(device=DEV)
  g.manual_seed((seed * 1000003 + sum(ord(c) * 31 ** i for i, c in enumerate(name))) % (1 << 62))
  return g


def _normal(seed, name, shape, sd=1.0, mean=0.0, dtype=torch.float32):
  return (torch.randn(*shape, generator=_gen(seed, name), device=DEV) * sd + mean).to(dtype)


def _whole(seed, name, lo, hi, shape, dtype=torch.int32):
  return torch.randint(lo, hi, shape, generator=_gen(seed, name), device=DEV, dtype=dtype)


def _weights(case, seed):
  """weights(name, shape) as Decoder takes them: matrices N(0, 0.02), norms near 1, in bf16 as checkpoints have them."""
  tied = MODELS[case["model"]]["tied"]
  def get(name, shape):
    if "norm" in name: return _normal(seed, name, shape, 0.1, 1.0, torch.bfloat16)
    return _normal(seed, name, shape, (0.1 if tied else 1.0) if name == "embed" else 0.02, 0.0, torch.bfloat16)
  return get


def _config(case, places):
  m = MODELS[case["model"]]
  return llama.model(layers=case["layers"], places=places, **m)


def _fill_cache(seed, name, cache):
  """Keys and values about N(0, 1): drawn in the cache's own type, a block float's magnitudes and exponents."""
  if isinstance(cache, ops.BfpCache):
    rows = cache.planes * cache.length
    mags = rows * cache.head_dim // (1 if cache.fmt == "bfp8" else 2)
    exps = rows * cache.head_dim // 16
    if cache.fmt == "bfp8": m = _whole(seed, name, -127, 128, (mags,), torch.int16).to(torch.uint8)
    else:
      lo, hi = _whole(seed, name, -7, 8, (mags,), torch.int16), _whole(seed, name + "'", -7, 8, (mags,), torch.int16)
      m = ((lo & 15) | (hi & 15) << 4).to(torch.uint8)
    cache.data[:mags].copy_(m)
    cache.data[cache.data.numel() - exps:].copy_(_whole(seed, name + "e", 126, 129, (exps,), torch.int16).to(torch.uint8))
  else: cache.normal_(generator=_gen(seed, name))


def _cache_values(cache):
  """A cache's values in 64 bits, [planes][length][head_dim]."""
  if not isinstance(cache, ops.BfpCache): return cache.double()
  rows, hd = cache.planes * cache.length, cache.head_dim
  exps = cache.data[cache.data.numel() - rows * hd // 16:].double()
  if cache.fmt == "bfp8": q, bias = cache.data[:rows * hd].view(torch.int8).double(), 133
  else:
    b = cache.data[:rows * hd // 2].to(torch.int16)
    q = torch.stack([b & 15, b >> 4], -1)
    q, bias = torch.where(q > 7, q - 16, q).double(), 129
  return (q.reshape(-1, 16) * torch.exp2(exps - bias)[:, None]).reshape(cache.planes, cache.length, hd)


def _row_places(last, batch):
  """Each row's place: from the last place down to half of it."""
  return [last - i * last // (2 * batch) for i in range(batch)]


def _moe_inputs(case, seed):
  dim, ffn = MOE[case["model"]]
  bf = torch.bfloat16
  return dict(x=_normal(seed, "x", (case["rows"], dim)), norm=_normal(seed, "norm", (dim,), 0.1, 1.0),
              router=_normal(seed, "router", (dim, EXPERTS), 0.02, 0.0, bf),
              gate_up=lambda e: _normal(seed, f"gate_up{e}", (dim, 2 * ffn), 0.02, 0.0, bf),
              down=lambda e: _normal(seed, f"down{e}", (ffn, dim), 0.02, 0.0, bf))


def _pack_parts(case, seed):
  dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
  if not case["parts"]: return [_normal(seed, "w", (case["K"], case["out"]), 0.02, 0.0, dt)]
  return [_normal(seed, f"w{i}", (case["out"], case["K"]), 0.02, 0.0, dt) for i in range(case["parts"])]


def prepare(case, seed):
  kind = case["kind"]
  if kind == "matmul":
    x = _normal(seed, "x", (case["rows"], case["K"]), dtype=torch.float32 if case["x"] == "fp32" or case["rows"] < 3 else torch.bfloat16)
    w = ops.pack(_normal(seed, "w", (case["K"], case["N"]), 0.02, 0.0, torch.bfloat16), case["fmt"])
    return dict(kind=kind, x=x, w=w, mm=ops.gemv if case["rows"] < 3 else ops.gemm)
  if kind == "decode":
    c = _config(case, case["cache"])
    dec = llama.Decoder(c, _weights(case, seed), mode=case["mode"], kv=case["kv"], batch=case["batch"], context=case["cache"], slots=case["batch"])
    for l, cache in enumerate(dec.cache): _fill_cache(seed, f"cache{l}", cache)
    return dict(kind=kind, dec=dec, ids=_whole(seed, "ids", 0, c.vocab, (case["batch"],)).tolist(),
                places=_row_places(case["place"], case["batch"]), slots=list(range(case["batch"])))
  if kind == "prefill":
    c = _config(case, case["p0"] + case["tokens"])
    dec = llama.Decoder(c, _weights(case, seed), mode=case["mode"], kv=case["kv"], context=case["p0"] + case["tokens"])
    for l, cache in enumerate(dec.cache): _fill_cache(seed, f"cache{l}", cache)
    return dict(kind=kind, dec=dec, p0=case["p0"], ids=_whole(seed, "ids", 0, c.vocab, (case["tokens"],)).tolist())
  if kind == "attend":
    h, kv, hd = HEADS[case["model"]]
    b, n = case["batch"], case["context"]
    cache = ops.kv_cache(2 * kv, b * n, hd, case["kv"], DEV)
    _fill_cache(seed, "cache", cache)
    q = _normal(seed, "q", (b, h * hd))
    return dict(kind=kind, q=q, cache=cache, heads=(h, kv, hd), context=n, o=torch.empty_like(q),
                places=torch.tensor(_row_places(n - 1, b), dtype=torch.int32, device=DEV),
                first=torch.arange(b, dtype=torch.int32, device=DEV) * n, ws=ops.attention_workspace(b, h, hd, n, DEV))
  if kind == "moe":
    i = _moe_inputs(case, seed)
    dim, ffn = MOE[case["model"]]
    # (an expert at a time: the experts' bf16 weights never lie in memory all at once)
    gu, dn = ([ops.pack(f(e), case["fmt"]) for e in range(EXPERTS)] for f in (i["gate_up"], i["down"]))
    cat = lambda ps, K, N: ops.BfpWeight(torch.cat([p.mant for p in ps]), torch.cat([p.exps for p in ps]), K, N, case["fmt"])
    ex = ops.Experts(cat(gu, dim, 2 * ffn), cat(dn, ffn, dim), EXPERTS, dim, ffn)
    ws = torch.empty(ops.lib.load().fh_moe_workspace_bytes(case["rows"], EXPERTS, ffn, dim), dtype=torch.uint8, device=DEV)
    ssq = i["x"].square().reshape(case["rows"], dim // 16, 16).sum(-1)  # (the matmul before the layer leaves these)
    return dict(kind=kind, x=i["x"], ssq=ssq, norm=i["norm"], router=i["router"], ex=ex, ws=ws)
  if kind == "tensor":
    rt = Runtime(0)
    def made(name, r, c, d):
      t = _normal(seed, name, (r, c), dtype=torch.bfloat16 if d == "bf16" else torch.float32).cpu()
      return Tensor.frombytes(rt, r, c, (t.view(torch.int16) if d == "bf16" else t).numpy().tobytes(), dtype=d)
    return dict(kind=kind, a=made("a", case["M"], case["K"], case["a"]), b=made("b", case["K"], case["N"], case["b"]))
  return dict(kind=kind, parts=_pack_parts(case, seed), rows=case["parts"] > 0, fmt=case["fmt"])


def run(s):
  kind = s["kind"]
  if kind == "matmul": return s["mm"](s["x"], s["w"])
  if kind == "decode":
    logits, picks = s["dec"].step(s["ids"], s["places"], s["slots"])
    # (a batch's picks follow from its logits: near ties between two tokens may fall either way)
    return dict(logits=logits, caches=_buffers(s["dec"]))
  if kind == "prefill":
    logits, pick = s["dec"].prefill(s["ids"], p0=s["p0"])
    return dict(logits=logits, caches=_buffers(s["dec"]))
  if kind == "attend":
    return ops.attention_decode(s["q"], s["cache"], *s["heads"], s["places"], s["first"], s["context"], s["ws"], o=s["o"])
  if kind == "moe":
    ids, weights, dense = ops.moe_route(s["x"], s["router"], EXPERTS, TOP, norm_w=s["norm"])
    return dict(ids=ids, weights=weights, out=ops.moe_experts(s["x"], s["ex"], dense, residual=s["x"], norm_w=s["norm"], ssq_in=s["ssq"], ws=s["ws"]))
  if kind == "tensor": return (s["a"] @ s["b"]).realize().data
  bw = ops.pack_parts(s["parts"], s["fmt"]) if s["rows"] else ops.pack(s["parts"][0], s["fmt"])
  return dict(mant=bw.mant, exps=bw.exps)


def _buffers(dec):
  """The first and the last block's cache (every block's go the same way; 64 outputs at most)."""
  got = [dec.cache[0], dec.cache[-1]]
  return [x.data if isinstance(x, ops.BfpCache) else x for x in got]


# ---- the work ----------------------------------------------------------------------------------------------------------
def _bits(fmt):  # bytes a value
  return {"bfp8": 17 / 16, "bfp4": 9 / 16, "bf16": 2, "fp32": 4}[fmt]


def _layer_mats(case):
  """(K, N, format) of a block's matrices, and of the output layer."""
  m = MODELS[case["model"]]
  h, kv, hd = HEADS[case["model"]]
  up = "bfp8" if case["mode"] == "bfp8" else "bfp4"
  down = "bfp4" if case["mode"] == "experts" else "bfp8"
  return [(m["dim"], (h + 2 * kv) * hd, "bfp8"), (h * hd, m["dim"], "bfp8"), (m["dim"], 2 * m["ffn"], up),
          (m["ffn"], m["dim"], down)], (m["dim"], m["vocab"], "bfp8")


def work(case):
  kind = case["kind"]
  if kind == "matmul":
    r, K, N = case["rows"], case["K"], case["N"]
    return {"bytes": K * N * _bits(case["fmt"]) + r * K * (4 if case["x"] == "fp32" or r < 3 else 2) + r * N * 4, "flops": 2 * r * K * N}
  if kind in ("decode", "prefill"):
    m, (h, kv, hd) = MODELS[case["model"]], HEADS[case["model"]]
    mats, head = _layer_mats(case)
    L = case["layers"]
    weights = sum(K * N * _bits(f) for K, N, f in mats) * L + head[0] * head[1] * _bits(head[2])
    per_row = sum(2 * K * N for K, N, f in mats) * L
    row = 2 * kv * hd * _bits(case["kv"])  # a cached token's bytes in a block
    if kind == "decode":
      seen = sum(p + 1 for p in _row_places(case["place"], case["batch"]))
      B = case["batch"]
      return {"bytes": weights + L * row * (seen + B) + B * (m["vocab"] * 4 + m["dim"] * 2),
              "flops": B * (per_row + 2 * head[0] * head[1]) + L * 4 * h * hd * seen}
    T, p0 = case["tokens"], case["p0"]
    pairs = T * p0 + T * (T + 1) // 2
    return {"bytes": weights + L * row * (p0 + T) + T * m["dim"] * 2 + m["vocab"] * 4,
            "flops": T * per_row + 2 * head[0] * head[1] + L * 4 * h * hd * pairs}
  if kind == "attend":
    h, kv, hd = HEADS[case["model"]]
    seen = sum(p + 1 for p in _row_places(case["context"] - 1, case["batch"]))
    return {"bytes": 2 * kv * hd * _bits(case["kv"]) * seen + case["batch"] * h * hd * 8, "flops": 4 * h * hd * seen}
  if kind == "moe":
    dim, ffn = MOE[case["model"]]
    r = case["rows"]
    touched = EXPERTS * (1 - (1 - TOP / EXPERTS) ** r)  # experts that some row picks, on average
    return {"bytes": touched * 3 * dim * ffn * _bits(case["fmt"]) + EXPERTS * dim * 2 + r * dim * 8,
            "flops": r * (TOP * 6 * dim * ffn + 2 * EXPERTS * dim)}
  if kind == "tensor":
    M, K, N = case["M"], case["K"], case["N"]
    return {"bytes": _bits(case["a"]) * (M * K + K * N + M * N), "flops": 2 * M * K * N}
  n = case["K"] * case["out"] * max(1, case["parts"])
  return {"bytes": n * (_bits(case["dtype"]) + _bits(case["fmt"])), "flops": 0}


def tolerance(case):
  """About four times the distance from exact(), as measured: fp32 sums of exact products 1e-7 (a single matmul), a
  batch-1 step's bf16 cache 1e-4, bf16 rows through a few blocks of a batched step 6e-3 and through up to 30 blocks of a
  prompt 1.2e-2, attention's fp32 softmax 4e-6, a mixture's bf16 rows 2.6e-3, a bf16 result's own rounding 1.7e-3."""
  kind = case["kind"]
  if kind == "pack": return "exact"
  if kind == "matmul": return {"rel": 1e-5, "max": 1e-4}
  if kind == "decode" and case["batch"] < 3: return {"rel": 1e-3, "max": 1e-2, "differ": 1e-3}
  if kind in ("decode", "prefill"): return {"rel": 2e-2 if kind == "decode" else 3e-2, "max": 0.3, "differ": 1e-3 if kind == "decode" else 1e-2}
  if kind == "attend": return {"rel": 2e-5, "max": 2e-4}
  if kind == "moe": return {"rel": 1e-2, "max": 5e-2}
  return {"rel": 7e-3, "max": 3e-2} if case["a"] == "bf16" else {"rel": 3e-5, "max": 3e-4}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------
def _bfp(w, fmt):
  """A matrix of bf16 values as the block float holds it, in 64 bits: runs of 16 along a row share their largest bf16
  exponent, each value 7 (bfp8) or 3 (bfp4) bits of magnitude rounded to nearest, ties up, and saturated."""
  b = w.to(torch.bfloat16).view(torch.int16).to(torch.int32).reshape(w.shape[0], -1, 16) & 0xFFFF
  e = b >> 7 & 255
  m = (b & 127) | torch.where(e != 0, 128, 0)
  top = e.amax(-1, keepdim=True)
  shift = (top - e).clamp(max=8)
  if fmt == "bfp8": q, bias = ((m + (1 << shift)) >> (shift + 1)).clamp(max=127), 133
  else:
    near = shift.clamp(max=3)
    q, bias = torch.where(shift < 4, ((m + (16 << near)) >> (near + 5)).clamp(max=7), 0), 129
  q = torch.where(b >> 15 != 0, -q, q)
  return (q.double() * torch.exp2((top - bias).double())).reshape(w.shape)


def _rms(x, w, eps):
  return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _tables(c, hd, places):
  """cos and sin by place, rounded to bf16 as the model's tables are."""
  inv = 1 / c.theta ** (np.arange(0, hd, 2, dtype=np.float32) / hd)
  a = np.arange(places, dtype=np.float32)[:, None] * inv[None]
  both = lambda f: torch.from_numpy(np.concatenate([f(a)] * 2, 1)).to(DEV).to(torch.bfloat16).double()
  return both(np.cos), both(np.sin)


def _rope(x, cos, sin):  # x [rows][heads][hd]
  half = x.shape[-1] // 2
  return x * cos[:, None] + torch.cat([-x[..., half:], x[..., :half]], -1) * sin[:, None]


def _attend(q, k, v, hd):
  """q [rows][heads][hd] over k, v [kv][keys][hd], row r of `rows` seeing all but the last rows - 1 - r keys."""
  rows, h, _ = q.shape
  kv, n, _ = k.shape
  out = torch.empty_like(q)
  late = torch.arange(n, device=q.device)[None] > (n - rows + torch.arange(rows, device=q.device))[:, None]
  for g in range(kv):
    s = q[:, g * (h // kv):(g + 1) * (h // kv)].permute(1, 0, 2).matmul(k[g].T.contiguous()) / math.sqrt(hd)
    out[:, g * (h // kv):(g + 1) * (h // kv)] = torch.softmax(s.masked_fill(late, -math.inf), -1).matmul(v[g]).permute(1, 0, 2)
  return out


def _forward(case, seed, places):
  """The model over the sequences' rows: places is each sequence's (places of its rows). Last rows' logits, and each
  block's cache values (sequence after sequence)."""
  c = _config(case, case["cache"] if case["kind"] == "decode" else case["p0"] + case["tokens"])
  h, kv, hd = HEADS[case["model"]]
  length, m = c.places, MODELS[case["model"]]
  get = _weights(case, seed)
  mats, headm = _layer_mats(case)
  rows = sum(len(p) for p in places)
  ids = _whole(seed, "ids", 0, c.vocab, (rows,)).long()
  x = get("embed", (c.vocab, c.dim))[ids].double()
  cos, sin = _tables(c, hd, length)
  at = torch.tensor([q for p in places for q in p], device=DEV)
  caches = []
  for l in range(c.layers):
    pre = f"layers.{l}."
    mat = dict(zip(("qkv_proj", "o_proj", "gate_up_proj", "down_proj"), mats))
    W = lambda n: _bfp(get(pre + n, mat[n][:2]), mat[n][2])
    cache = ops.kv_cache(2 * kv, len(places) * length, hd, case["kv"], DEV)
    _fill_cache(seed, f"cache{l}", cache)
    cv = _cache_values(cache)
    n = _rms(x, get(pre + "input_layernorm", (1, c.dim)).double(), c.eps)
    qkv = (n @ W("qkv_proj")).reshape(rows, h + 2 * kv, hd)
    q, k, v = _rope(qkv[:, :h], cos[at], sin[at]), _rope(qkv[:, h:h + kv], cos[at], sin[at]), qkv[:, h + kv:]
    o, r = torch.empty_like(q), 0
    for s, p in enumerate(places):
      a, b = s * length, s * length + p[-1] + 1
      cv[:kv, a + p[0]:b] = k[r:r + len(p)].permute(1, 0, 2)
      cv[kv:, a + p[0]:b] = v[r:r + len(p)].permute(1, 0, 2)
      o[r:r + len(p)] = _attend(q[r:r + len(p)], cv[:kv, a:b], cv[kv:, a:b], hd)
      r += len(p)
    caches.append(cv if l in (0, c.layers - 1) else None)
    x = x + o.reshape(rows, h * hd) @ W("o_proj")
    n = _rms(x, get(pre + "post_attention_layernorm", (1, c.dim)).double(), c.eps)
    gu = n @ W("gate_up_proj")
    x = x + (torch.nn.functional.silu(gu[:, :c.ffn]) * gu[:, c.ffn:]) @ W("down_proj")
  last = torch.tensor([sum(len(p) for p in places[:s + 1]) - 1 for s in range(len(places))], device=DEV)
  n = _rms(x[last], get("norm", (1, c.dim)).double(), c.eps)
  head = get("embed", (c.vocab, c.dim)).T.contiguous() if m["tied"] else get("embed.T", (c.dim, c.vocab))
  logits = torch.cat([n @ _bfp(p, headm[2]) for p in head.split(16384, 1)], 1)
  # (a block-float cache's outputs are its packed bytes)
  return dict(logits=logits, caches=[caches[0], caches[-1]] if case["kv"] in ("bf16", "fp32") else [None, None])


def exact(case, seed):
  kind = case["kind"]
  if kind == "matmul":
    x = _normal(seed, "x", (case["rows"], case["K"]), dtype=torch.float32 if case["x"] == "fp32" or case["rows"] < 3 else torch.bfloat16)
    return x.double() @ _bfp(_normal(seed, "w", (case["K"], case["N"]), 0.02, 0.0, torch.bfloat16), case["fmt"])
  if kind == "decode": return _forward(case, seed, [[p] for p in _row_places(case["place"], case["batch"])])
  if kind == "prefill": return _forward(case, seed, [list(range(case["p0"], case["p0"] + case["tokens"]))])
  if kind == "attend":
    h, kv, hd = HEADS[case["model"]]
    b, n = case["batch"], case["context"]
    cache = ops.kv_cache(2 * kv, b * n, hd, case["kv"], DEV)
    _fill_cache(seed, "cache", cache)
    q = _normal(seed, "q", (b, h * hd)).double().reshape(b, h, hd)
    cv = _cache_values(cache)
    return torch.cat([_attend(q[r:r + 1], cv[:kv, r * n:r * n + p + 1], cv[kv:, r * n:r * n + p + 1], hd)
                      for r, p in enumerate(_row_places(n - 1, b))]).reshape(b, h * hd)
  if kind == "moe":
    i = _moe_inputs(case, seed)
    dim, ffn = MOE[case["model"]]
    n = _rms(i["x"].double(), i["norm"].double(), 1e-5)
    best = (n @ i["router"].double()).topk(TOP, -1)
    weights, out = torch.softmax(best.values, -1), i["x"].double()
    for e in range(EXPERTS):
      row, k = (best.indices == e).nonzero(as_tuple=True)
      if not len(row): continue
      gu = n[row] @ _bfp(i["gate_up"](e), case["fmt"])
      out[row] += weights[row, k][:, None] * ((torch.nn.functional.silu(gu[:, :ffn]) * gu[:, ffn:]) @ _bfp(i["down"](e), case["fmt"]))
    return dict(ids=None, weights=weights, out=out)
  if kind == "tensor":
    made = lambda name, r, c, d: _normal(seed, name, (r, c), dtype=torch.bfloat16 if d == "bf16" else torch.float32).double()
    return (made("a", case["M"], case["K"], case["a"]) @ made("b", case["K"], case["N"], case["b"]))[None]
  return None
