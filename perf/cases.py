"""Performance cases: what users of this library have it do, over the range of sizes, types and directions it serves.

Every case is one pass through the public entry points (`ragged_dot`, `ragged_gather`, `ragged_gather_reduce`,
`gated_linear_unit`, `AsQArray`) on inputs a program would hold anyway. `path` says which:

  dot    one `ragged_dot` over expert weights in the form `weights` names (plain, or quantised the usual ways), with the
         activations as they come or quantised on the fly in the form `quantise` names
  train  a training step's `ragged_dot`: forward, then the gradients of both operands
  ffn    an MoE layer's expert block: tokens permuted into expert order, gate-up product with silu, down product, and the
         weighted combine back into token order
  glu    the dense `gated_linear_unit` (shared expert, dense layer)

Rows reach their experts through a top-k router; `skew` is the exponent of the experts' Zipf popularity (0: all alike).
"""

import math

import torch

import tokamax_amd
from tokamax_amd import AsQArray, QArray

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_BYTES = {"bf16": 2, "f16": 2, "f32": 4}
# Bytes of one weight, and k rows that share a scale (0: one scale per (group, column)), by form.
_WEIGHTS = {"plain": (None, None), "int8": (1, 0), "int4_k128": (0.5, 128), "fp8": (1, 0), "fp8_128x128": (1, 128)}


def listed():
  return [
      # One decoding step's product of a 128-expert layer: 32 sequences, 8 experts each, int8 weights.
      dict(name="decode_int8", path="dot", tokens=32, top_k=8, groups=128, k=2048, n=768, dtype="bf16", weights="int8",
           quantise="none", skew=0.0),
      # The whole expert block of the same layer for four sequences: the smallest call, bound by latency and launches.
      dict(name="decode_ffn", path="ffn", tokens=4, top_k=8, groups=128, k=2048, n=768, dtype="bf16", skew=0.0),
      # A server that batches 96 sequences over int4 weights (scales per 128 k rows): between decode and prefill.
      dict(name="batch_int4", path="dot", tokens=96, top_k=2, groups=8, k=4096, n=14336, dtype="bf16", weights="int4_k128",
           quantise="none", skew=0.0),
      # Prefill of 8192 tokens through the expert block of an 8-expert layer: the largest call.
      dict(name="prefill_ffn", path="ffn", tokens=8192, top_k=2, groups=8, k=4096, n=14336, dtype="bf16", skew=0.0),
      # Prefill of a 256-expert layer with popular and hardly used experts.
      dict(name="prefill_many_experts", path="dot", tokens=8192, top_k=8, groups=256, k=7168, n=2048, dtype="bf16",
           weights="plain", quantise="none", skew=1.0),
      # A short prompt with sizes that fit no tile.
      dict(name="prefill_odd", path="dot", tokens=777, top_k=4, groups=24, k=1416, n=2824, dtype="f16", weights="plain",
           quantise="none", skew=0.5),
      # fp8 with block scales (1 x 128 activations, 128 x 128 weights) on a 32-expert shard, quantised on the way in.
      dict(name="prefill_fp8_blocks", path="dot", tokens=2048, top_k=4, groups=32, k=7168, n=2048, dtype="bf16",
           weights="fp8_128x128", quantise="fp8_k128", skew=0.5),
      # Activations quantised to fp8 per row on the way in, fp8 weights with one scale per column.
      dict(name="prefill_fp8", path="dot", tokens=4096, top_k=2, groups=8, k=4096, n=14336, dtype="bf16", weights="fp8",
           quantise="fp8", skew=0.0),
      # A training step's product in an 8-expert layer: 2048 tokens.
      dict(name="train", path="train", tokens=2048, top_k=2, groups=8, k=4096, n=14336, dtype="bf16", skew=0.0),
      # ... and in a layer of 128 small experts.
      dict(name="train_many_experts", path="train", tokens=4096, top_k=8, groups=128, k=2048, n=768, dtype="bf16", skew=0.5),
      # Single precision, forward and gradients, at the size of a numerical study.
      dict(name="train_f32", path="train", tokens=512, top_k=2, groups=8, k=512, n=1024, dtype="f32", skew=0.0),
      # The dense gated unit for a batch of 256 tokens.
      dict(name="glu", path="glu", tokens=256, k=4096, n=14336, dtype="bf16"),
  ]


def _log_int(rng, lo, hi, step=1):
  """A multiple of `step` between lo and hi, spread over the logarithm."""
  x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
  return max(-(-lo // step) * step, min(hi // step * step, int(round(x / step)) * step))


def _draw_once(rng):
  path = rng.choice(("dot", "dot", "dot", "train", "train", "ffn", "glu"))
  if path == "glu":
    return dict(path=path, tokens=_log_int(rng, 1, 8192), k=_log_int(rng, 512, 8192, 64), n=_log_int(rng, 512, 16384, 32),
                dtype=rng.choice(("bf16", "bf16", "f16")))
  groups = rng.choice((8, 16, 24, 32, 64, 128, 256))
  case = dict(path=path, tokens=_log_int(rng, 1, 16384), top_k=rng.choice((1, 2, 4, 8)), groups=groups,
              k=_log_int(rng, 512, 8192, 8), n=_log_int(rng, 512, 16384, 8), dtype="bf16",
              skew=rng.choice((0.0, 0.5, 1.0)))
  if path == "ffn":
    case.update(k=_log_int(rng, 512, 8192, 64), n=_log_int(rng, 512, 16384, 64))
  elif path == "train":
    case.update(tokens=_log_int(rng, 64, 16384), dtype=rng.choice(("bf16", "bf16", "f16", "f32")))
  else:
    weights = rng.choice(("plain", "plain", "int8", "int4_k128", "fp8", "fp8_128x128"))
    quantise = {"fp8": "fp8", "fp8_128x128": "fp8_k128"}.get(weights, "none")
    if weights == "int4_k128":
      quantise = rng.choice(("none", "fp8"))
    case.update(weights=weights, quantise=quantise)
    if weights == "plain":
      case.update(dtype=rng.choice(("bf16", "bf16", "f16", "f32")))
    else:
      # (quantised operands come with k a multiple of the scale blocks and the row counts the quantisers take)
      case.update(k=_log_int(rng, 512, 8192, 128), n=_log_int(rng, 512, 16384, 128 if weights == "fp8_128x128" else 16))
      if quantise != "none":
        case.update(tokens=_log_int(rng, 64, 16384, 4))
  return case


def _cost(case):
  w = work(case)
  rate = 1e14 if case["dtype"] == "f32" else 1e15
  return w["bytes"] / 4e12 + w["flops"] / rate


def _footprint(case):
  """Bytes of expert weights in the type they are drawn in (all experts are resident, used or not)."""
  matrices = {"ffn": 3, "glu": 2, "train": 2}.get(case["path"], 1)
  return matrices * case.get("groups", 1) * case["k"] * case["n"] * _BYTES[case["dtype"]]


def draw(rng):
  limit = max(_cost(c) for c in listed())
  while True:
    case = _draw_once(rng)
    if _cost(case) <= 0.9 * limit and _footprint(case) <= 12e9:
      return case


def _touched(case):
  """Experts that get at least one row, on average."""
  if case["path"] == "glu":
    return 1.0
  groups, tokens, top_k = case["groups"], case["tokens"], case["top_k"]
  p = [(i + 1.0) ** -case["skew"] for i in range(groups)]
  total = sum(p)
  return sum(1.0 - (1.0 - min(1.0, top_k * x / total)) ** tokens for x in p)


def work(case):
  k, n, b = case["k"], case["n"], _BYTES[case["dtype"]]
  tokens = case["tokens"]
  if case["path"] == "glu":
    return dict(bytes=(tokens * k + 2 * k * n + tokens * n) * b, flops=4 * tokens * k * n)
  rows, touched = tokens * case["top_k"], _touched(case)
  if case["path"] == "ffn":
    return dict(bytes=(2 * tokens * k + touched * 3 * k * n) * b, flops=6 * rows * k * n)
  if case["path"] == "train":
    # forward reads lhs and rhs and writes out; the gradients read dout and write both (lhs and rhs stay one read)
    return dict(bytes=(2 * rows * k + 2 * rows * n + touched * k * n + case["groups"] * k * n) * b, flops=6 * rows * k * n)
  wbytes, block = _WEIGHTS[case["weights"]]
  scales = 0
  if wbytes is None:
    wbytes = b
  else:
    columns = n // 128 if case["weights"] == "fp8_128x128" else n
    scales = 4 * columns * (k // block if block else 1)
  return dict(bytes=rows * k * b + touched * (k * n * wbytes + scales) + rows * n * b, flops=2 * rows * k * n)


def _generator(seed):
  return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, shape, std, dtype):
  return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)


def _route(case, gen):
  """Expert of every (token, choice): the top k of Gumbel-perturbed log-popularities, which are dealt out at random."""
  groups = case["groups"]
  rank = torch.randperm(groups, device="cuda", generator=gen).float() + 1.0
  noise = -torch.log(-torch.log(torch.rand(case["tokens"], groups, device="cuda", generator=gen).clamp_(1e-9, 1 - 1e-7)))
  expert = torch.topk(noise - case["skew"] * torch.log(rank), case["top_k"], dim=1).indices.reshape(-1)
  return expert, torch.bincount(expert, minlength=groups).to(torch.int32)


def _weights(case, gen):
  groups, k, n, form = case["groups"], case["k"], case["n"], case.get("weights", "plain")
  if form == "plain":
    return _normal(gen, (groups, k, n), k ** -0.5, _DTYPES[case["dtype"]])
  # A few experts at a time, so that the 16-bit originals of a large layer are never all there at once.
  parts = []
  qtype = {"int8": torch.int8, "int4_k128": torch.int4}.get(form, torch.float8_e4m3fn)
  tiled = {"int4_k128": {0: 1, 1: 128, 2: 1}, "fp8_128x128": {0: 1, 1: 128, 2: 128}}.get(form, {0: 1, 1: k, 2: 1})
  step = max(1, int(1e9 // (k * n * 2)))
  for g in range(0, groups, step):
    w = _normal(gen, (min(step, groups - g), k, n), k ** -0.5, torch.bfloat16)
    q = AsQArray(w, qtype, tiled_axes=tiled).as_qarray()
    parts.append(tokamax_amd.pack_int4(q) if form == "int4_k128" else q)
  return QArray(torch.cat([q.qvalue for q in parts]), torch.cat([q.scale for q in parts]), None, parts[0].qtype)


def prepare(case, seed):
  gen = _generator(seed)
  path, tokens, k, n, dtype = case["path"], case["tokens"], case["k"], case["n"], _DTYPES[case["dtype"]]
  state = dict(case=dict(case))
  if path == "glu":
    state["x"] = _normal(gen, (tokens, k), 1.0, dtype)
    state["w"] = _normal(gen, (k, 2, n), k ** -0.5, dtype)
    return state
  expert, state["group_sizes"] = _route(case, gen)
  rows = tokens * case["top_k"]
  if path == "ffn":
    order = torch.argsort(expert, stable=True)
    state["token_of_row"] = (order // case["top_k"]).to(torch.int32)
    state["row_of_slot"] = torch.argsort(order).to(torch.int32)
    state["gate"] = torch.rand(rows, device="cuda", generator=gen)
    state["valid"] = torch.ones(rows, dtype=torch.bool, device="cuda")
    state["h"] = _normal(gen, (tokens, k), 1.0, dtype)
    state["gate_up"] = _normal(gen, (case["groups"], k, 2 * n), k ** -0.5, dtype)
    state["down"] = _normal(gen, (case["groups"], n, k), n ** -0.5, dtype)
    return state
  state["lhs"] = _normal(gen, (rows, k), 1.0, dtype)
  state["rhs"] = _weights(case, gen)
  if path == "train":
    state["dout"] = _normal(gen, (rows, n), 1.0, dtype)
    state["lhs"].requires_grad_(True)
    state["rhs"].requires_grad_(True)
  return state


def run(state):
  case = state["case"]
  path = case["path"]
  if path == "glu":
    return tokamax_amd.gated_linear_unit(state["x"], state["w"], activation=torch.nn.functional.silu)
  group_sizes = state["group_sizes"]
  if path == "ffn":
    x = tokamax_amd.ragged_gather(state["h"], state["token_of_row"], 0, case["tokens"])
    y = _FFN_OP(x, state["gate_up"], group_sizes=group_sizes, fuse_gateup_activation="silu")
    z = tokamax_amd.ragged_dot(y, state["down"], group_sizes)
    return tokamax_amd.ragged_gather_reduce(z, state["row_of_slot"], state["gate"], state["valid"], case["top_k"])
  if path == "train":
    out = tokamax_amd.ragged_dot(state["lhs"], state["rhs"], group_sizes)
    dlhs, drhs = torch.autograd.grad(out, (state["lhs"], state["rhs"]), state["dout"])
    return dict(out=out, dlhs=dlhs, drhs=drhs)
  lhs = state["lhs"]
  if case["quantise"] == "fp8":
    lhs = AsQArray(lhs, torch.float8_e4m3fn, channelwise_axes=(0,))
  elif case["quantise"] == "fp8_k128":
    lhs = AsQArray(lhs, torch.float8_e4m3fn, channelwise_axes=(0,), tiled_axes={1: 128})
  out_dtype = None if case["weights"] == "plain" else _DTYPES[case["dtype"]]
  return tokamax_amd.ragged_dot(lhs, state["rhs"], group_sizes, preferred_element_type=out_dtype)


# The gate-up product is the operator's own argument (`ragged_dot` has no parameter for it).
_FFN_OP = tokamax_amd.HipRaggedDot()


def tolerance(case):
  """About four times the error measured against the same sums in 64 bits on the same (quantised) operands: 1.66e-3 for one
  product with a bf16 result (2.3e-3 where weights times their block scales are rounded to bf16 on the way in), 2.9e-3 for
  the three roundings of the expert block, 2.1e-4 for f16, 4e-7 to 6e-7 for f32 contractions of 500 to 1000 (growing with
  the root of the length: 1e-5 covers the longest)."""
  if case["dtype"] == "f32":
    return dict(rel=1e-5)
  if case["dtype"] == "f16":
    return dict(rel=1e-3)
  if case["path"] == "ffn":
    return dict(rel=1.2e-2)
  return dict(rel=1e-2 if case.get("weights", "").startswith("int4") else 7e-3)
