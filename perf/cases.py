"""The work that users of baretile_amd have it do, as cases to time and to compare.

Each case goes through the public surface: the Tensor API (eager, as a program that builds and realizes expressions
runs it), the Llama functions, and, for the decode steps that a serving loop repeats, a tensor.Recording of them
replayed. Shapes come from the repository's benchmark, tests and model configurations, or are generic.

Kinds:
  step    one decode step of a small Llama (the SmolLM-135M shapes of models.llama.smol), replayed: one token on the
          fused row kernels, or a batch of slots with its greedy heads as models.serve.Engine decodes it;
  slots   one block of a batched decode step (models.llama.slots_layer), every slot with a cache of its own, replayed;
  block   one block of a prompt's prefill (models.llama.layer), eager, from an empty cache or behind cached rows;
  attend  Tensor.attend alone: a decode step's over several layers' caches, replayed, or a prompt's, eager;
  linear  x @ W with W by columns and the elementwise tree above it as the epilogue: eager, or a decode step's several
          matrices, replayed;
  pack    a weight's way in and out: cast to a block float, columns(), and read back as bf16;
  norm    layernorm or softmax through the lazy graph, eager.
"""
import math

import numpy as np
import torch

from baretile_amd.models import llama, serve
from baretile_amd.runtime import Runtime
from baretile_amd.tensor import Recording, Tensor

SMOL = {"kind": "step", "dim": 576, "heads": 9, "kv": 3, "layers": 30, "ffn": 1536, "vocab": 49152}
LLAMA_8B = {"dim": 4096, "heads": 32, "kv": 8, "head": 128, "ffn": 14336}
THETA = 10000.0
EPS = 1e-5


def listed():
  return [
    # a chat's next token from the small model: one row through 30 layers, latency and launches
    {"name": "token_step", **SMOL, "fmt": "bfp8", "slots": 0, "size": 512, "at": 300},
    # the serving engine's step: 8 streams at places of their own in one shared cache, with their greedy heads
    {"name": "slots_step", **SMOL, "fmt": "bfp8", "slots": 8, "size": 512, "at": 300},
    # a large model's batched decode: 32 streams, 4096 cached rows each, bfp4 projections
    {"name": "block_decode_32", "kind": "slots", **LLAMA_8B, "slots": 32, "size": 4096, "fmt": "bfp4"},
    # a long prompt's prefill through one large block
    {"name": "block_prefill_2048", "kind": "block", **LLAMA_8B, "tokens": 2048, "start": 0, "size": 2048,
     "fmt": "bfp4"},
    # a short, ragged chunk of a prompt behind cached rows, bfp8 projections
    {"name": "block_prefill_ragged", "kind": "block", **LLAMA_8B, "tokens": 333, "start": 500, "size": 1024,
     "fmt": "bfp8"},
    # one stream's decode attention over a medium context, 8 layers' caches one after another
    {"name": "attend_decode_1", "kind": "attend", "heads": 32, "kv": 8, "head": 128, "batch": 1, "rows": 1,
     "keys": 4096, "cache": "bf16", "layers": 8, "ragged": False},
    # a batch of streams of uneven lengths on block-float caches
    {"name": "attend_decode_8_bfp8", "kind": "attend", "heads": 32, "kv": 8, "head": 128, "batch": 8, "rows": 1,
     "keys": 8191, "cache": "bfp8", "layers": 2, "ragged": True},
    # a long prompt's causal attention alone
    {"name": "attend_prefill", "kind": "attend", "heads": 32, "kv": 8, "head": 128, "batch": 1, "rows": 4096,
     "keys": 4096, "cache": "bf16", "layers": 1, "ragged": False},
    # the output layer of the small model at batch 1, over enough matrices that each is read from HBM
    {"name": "gemv_24", "kind": "linear", "m": 1, "k": 576, "n": 49152, "fmt": "bfp4", "act": "none", "layers": 24},
    # the smallest call: one fused product, realized at once
    {"name": "relu_small", "kind": "linear", "m": 128, "k": 576, "n": 1536, "fmt": "bfp8", "act": "relu", "layers": 1},
    # loading a large projection, and reading it back
    {"name": "pack_bfp4", "kind": "pack", "rows": 4096, "cols": 14336, "fmt": "bfp4"},
    # a normalization through the lazy graph
    {"name": "layernorm", "kind": "norm", "op": "layernorm", "batch": 1, "rows": 2048, "cols": 4096, "dtype": "bf16"},
  ]


def _log_int(rng, lo, hi):
  """An integer from lo to hi, spread over its logarithm."""
  return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
  kind = rng.choice(("step", "slots", "block", "block", "attend", "attend", "linear", "linear", "pack", "norm"))
  if kind == "step":
    kv, rep = rng.choice(((3, 3), (2, 4), (4, 1), (5, 3), (4, 3), (8, 1)))
    size = _log_int(rng, 64, 512)
    return {"kind": "step", "dim": 64 * kv * rep, "heads": kv * rep, "kv": kv, "layers": _log_int(rng, 2, 30),
            "ffn": 64 * _log_int(rng, 8, 40), "vocab": 256 * _log_int(rng, 8, 192), "fmt": rng.choice(("bfp8", "bfp4", "bf16")),
            "slots": rng.choice((0, 0, _log_int(rng, 2, 16))), "size": size, "at": rng.randint(size // 4, size - 2)}
  if kind in ("slots", "block"):
    kv, rep, hd = rng.choice(((8, 4, 128), (4, 4, 128), (8, 2, 128), (8, 4, 64), (5, 5, 64)))
    case = {"kind": kind, "dim": 256 * rng.randint(4, 16), "heads": kv * rep, "kv": kv, "head": hd,
            "ffn": 256 * _log_int(rng, 8, 56), "fmt": rng.choice(("bfp8", "bfp4", "bf16"))}
    if kind == "slots": return {**case, "slots": _log_int(rng, 5, 32), "size": _log_int(rng, 100, 4096)}
    tokens, start = _log_int(rng, 33, 2048), rng.choice((0, _log_int(rng, 1, 2000)))
    return {**case, "tokens": tokens, "start": start, "size": tokens + start + rng.randint(0, 100)}
  if kind == "attend":
    kv, rep, hd = rng.choice(((8, 4, 128), (3, 3, 64), (8, 8, 128), (4, 7, 64), (8, 1, 64), (2, 4, 128)))
    if rng.random() < 0.5:  # a decode step
      batch, keys = _log_int(rng, 1, 16), _log_int(rng, 50, 16384)
      layers = min(rng.randint(2, 8), 1 + 2 ** 31 // (batch * kv * keys * hd * 4))
      return {"kind": "attend", "heads": kv * rep, "kv": kv, "head": hd, "batch": batch, "rows": 1, "keys": keys,
              "cache": rng.choice(("bf16", "bf16", "bfp8", "bfp4")), "layers": layers, "ragged": rng.random() < 0.5}
    rows = _log_int(rng, 65, 4096)
    return {"kind": "attend", "heads": kv * rep, "kv": kv, "head": hd, "batch": 1, "rows": rows,
            "keys": rows + rng.choice((0, _log_int(rng, 1, 2048))), "cache": rng.choice(("bf16", "bf16", "bfp8")),
            "layers": 1, "ragged": False}
  if kind == "linear":
    fmt = rng.choice(("bfp8", "bfp4", "bf16"))
    act = rng.choice(("none", "relu", "silu", "residual"))
    if rng.random() < 0.4:  # a decode step's matrices
      k, n = 64 * _log_int(rng, 4, 64), 16 * _log_int(rng, 32, 3072)
      return {"kind": "linear", "m": _log_int(rng, 1, 16), "k": k, "n": n, "fmt": fmt, "act": act,
              "layers": min(rng.randint(4, 24), 2 + 2 ** 31 // (k * n * 2))}
    return {"kind": "linear", "m": _log_int(rng, 17, 4096), "k": rng.choice((64 * _log_int(rng, 2, 96), _log_int(rng, 100, 6000))),
            "n": _log_int(rng, 64, 8192), "fmt": fmt, "act": act, "layers": 1}
  if kind == "pack":
    return {"kind": "pack", "rows": _log_int(rng, 64, 8192), "cols": _log_int(rng, 64, 16384), "fmt": rng.choice(("bfp8", "bfp4"))}
  return {"kind": "norm", "op": rng.choice(("layernorm", "softmax")), "batch": rng.choice((1, 1, _log_int(rng, 2, 16))),
          "rows": _log_int(rng, 16, 2048), "cols": _log_int(rng, 64, 8192), "dtype": rng.choice(("bf16", "fp32"))}


# ---- inputs, as torch tensors made on the GPU from the seed alone

def _normal(g, *shape, scale=1.0, mean=0.0, dtype=torch.bfloat16):
  return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(scale).add_(mean).to(dtype)


def _tables(heads, kv, hd, places):
  """(cos, sin) bf16 rows as models.llama.rotary lays them out: q's heads scaled, then k's, then v's left as they are."""
  inv = (1 / THETA ** (np.arange(0, hd, 2, dtype=np.float32) / hd)).astype(np.float32)
  angles = np.asarray(places, np.float32)[:, None] * inv[None]
  cos, sin = (torch.from_numpy(np.concatenate([f(angles)] * 2, 1).astype(np.float32)).cuda() for f in (np.cos, np.sin))
  wide = lambda t, still: torch.cat([t * np.float32(hd ** -0.5)] * heads + [t] * kv + [torch.full_like(t, still)] * kv, 1).bfloat16()
  return wide(cos, 1.0), wide(sin, 0.0)


def _block_weights(g, case, hd):
  d, f, q, kv = case["dim"], case["ffn"], case["heads"] * hd, case["kv"] * hd
  return {"input_layernorm": _normal(g, 1, d, scale=0.1, mean=1.0), "post_attention_layernorm": _normal(g, 1, d, scale=0.1, mean=1.0),
          "qkv_proj": _normal(g, d, q + 2 * kv, scale=0.02), "o_proj": _normal(g, q, d, scale=0.02),
          "gate_up_proj": _normal(g, d, 2 * f, scale=0.02), "down_proj": _normal(g, f, d, scale=0.02)}


def _inputs(case, seed):
  g = torch.Generator("cuda").manual_seed(int(seed))
  kind, out = case["kind"], {}
  if kind == "step":
    hd, n = case["dim"] // case["heads"], max(1, case["slots"])
    out["layers"] = [_block_weights(g, case, hd) for _ in range(case["layers"])]
    out["norm"] = _normal(g, 1, case["dim"], scale=0.1, mean=1.0)
    out["embed"] = _normal(g, case["vocab"], case["dim"])
    out["caches"] = [_normal(g, 2 * case["kv"], n * case["size"], hd, scale=0.5) for _ in range(case["layers"])]
    out["ids"] = torch.randint(0, case["vocab"], (n,), generator=g, device="cuda", dtype=torch.int32)
    out["places"] = torch.randint(case["at"] // 2, case["at"] + 1, (n,), generator=g, device="cuda", dtype=torch.int32)
    if not case["slots"]: out["places"].fill_(case["at"])
  elif kind in ("slots", "block"):
    out["weights"] = _block_weights(g, case, case["head"])
    n = case["slots"] if kind == "slots" else case["tokens"]
    out["x"] = _normal(g, n, case["dim"], dtype=torch.float32)
    if kind == "slots":
      out["then"] = _normal(g, 1, case["dim"], scale=0.1, mean=1.0)
      out["keys"], out["values"] = (_normal(g, n * case["kv"], case["size"], case["head"]) for _ in range(2))
    else:
      out["cache"] = torch.zeros(2 * case["kv"], case["size"], case["head"], device="cuda", dtype=torch.bfloat16)
      if case["start"]: out["cache"][:, :case["start"]] = _normal(g, 2 * case["kv"], case["start"], case["head"])
  elif kind == "attend":
    b, r = case["batch"], case["rows"]
    shape = (b * case["kv"], case["keys"], case["head"])
    out["q"] = [_normal(g, b * case["heads"], r, case["head"], scale=case["head"] ** -0.5) for _ in range(case["layers"])]
    out["k"] = [_normal(g, *shape) for _ in range(case["layers"])]
    out["v"] = [_normal(g, *shape) for _ in range(case["layers"])]
    last = torch.arange(case["keys"] - r, case["keys"], device="cuda", dtype=torch.int32).repeat(b, 1)
    if case["ragged"]:
      last -= torch.randint(0, case["keys"] // 2, (b, 1), generator=g, device="cuda", dtype=torch.int32)
    out["places"] = last.clamp_(min=0).repeat_interleave(case["heads"], 0)[:, :, None]
  elif kind == "linear":
    out["x"] = _normal(g, case["m"], case["k"])
    out["w"] = [_normal(g, case["k"], case["n"], scale=0.02) for _ in range(case["layers"])]
    if case["act"] == "residual": out["r"] = _normal(g, case["m"], case["n"], dtype=torch.float32)
  elif kind == "pack":
    out["w"] = _normal(g, case["rows"], case["cols"], scale=0.02)
  else:
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    out["x"] = _normal(g, case["batch"], case["rows"], case["cols"], dtype=dtype)
    if case["op"] == "layernorm":
      out["w"], out["b"] = _normal(g, 1, case["cols"], scale=0.1, mean=1.0, dtype=dtype), _normal(g, 1, case["cols"], dtype=dtype)
  return out


# ---- tensors between torch and the runtime

_rt = None


def _runtime():
  global _rt
  if _rt is None or _rt.closed: _rt = Runtime()
  return _rt


NAMES = {torch.bfloat16: "bf16", torch.float32: "fp32", torch.int32: "int32"}


def _tensor(t):
  """A torch tensor of up to three dimensions as a Tensor, copied on the device."""
  rt, t = _runtime(), t.contiguous()
  shape = (1,) * (3 - t.dim()) + tuple(t.shape)
  out = Tensor(rt, shape[1], shape[2], batch=shape[0], dtype=NAMES[t.dtype])
  torch.cuda.synchronize()
  rt.copy(out.addr, t.data_ptr(), t.numel() * t.element_size())
  rt.wait()
  return out


class _Shared:
  """A realized, contiguous Tensor's memory for torch to read in place; it keeps the tensor."""
  KINDS = {"bf16": "<i2", "fp32": "<f4", "int32": "<i4"}

  def __init__(self, t):
    self.tensor = t
    self.__cuda_array_interface__ = {"shape": t.shape, "typestr": self.KINDS[t.dtype], "data": (t.addr, False), "version": 2}


def _torch(t):
  v = torch.as_tensor(_Shared(t), device="cuda")
  return v.view(torch.bfloat16) if t.dtype == "bf16" else v


def _columns(w, fmt):
  t = _tensor(w)
  return (t.cast(fmt) if fmt != "bf16" else t).columns()


def _replayed(fn):
  """fn, run once, then recorded: the recording and what it writes, as torch tensors."""
  rt = _runtime()
  fn()
  rt.wait()
  rec = Recording(rt)
  with rec: out = fn()
  return rec, [_torch(t) for t in out]


def _config(case, hd):
  return llama.model(dim=case["dim"], heads=case["heads"], kv=case["kv"], layers=case.get("layers", 1), eps=EPS,
                     theta=THETA, vocab=case.get("vocab"), ffn=case["ffn"], head_dim=hd)


def _upload_block(weights, fmt):
  return {k: _columns(v, fmt) if k.endswith("_proj") else _tensor(v) for k, v in weights.items()}


def prepare(case, seed):
  x, kind, s = _inputs(case, seed), case["kind"], {"case": case}
  if kind == "step":
    hd = case["dim"] // case["heads"]
    c, fmt = _config(case, hd), case["fmt"]
    w = {f"layers.{l}.{k}": t for l, p in enumerate(x["layers"]) for k, t in _upload_block(p, fmt).items()}
    w["norm"], w["embed"], w["embed.T"] = _tensor(x["norm"]), _tensor(x["embed"]), _columns(x["embed"].T, fmt)
    both = _tensor(torch.cat(_tables(case["heads"], case["kv"], hd, np.arange(case["size"])), 1))
    n = both.cols // 2
    w["cos_sin"], w["cos"], w["sin"], w["turn"] = both, both[:, :n], both[:, n:], None
    ids, places, caches = _tensor(x["ids"][None]), _tensor(x["places"][None]), [_tensor(t) for t in x["caches"]]
    if case["slots"]:
      def step():
        logits = llama.forward(ids, places, w, c, caches, slots=case["slots"]).realize()
        return [logits, *serve.heads(logits, k=1)]
    else:
      def step(): return [llama.forward(ids, places, w, c, caches).realize()]
    s["keep"] = (w, ids, places)
    s["rec"], s["out"] = _replayed(step)
    s["out"] += [_torch(t) for t in caches]
  elif kind == "slots":
    c, p = _config(case, case["head"]), _upload_block(x["weights"], case["fmt"])
    xs, keys, values, then = (_tensor(x[k]) for k in ("x", "keys", "values", "then"))
    place = case["size"] - 1
    rot = [_tensor(t) for t in _tables(case["heads"], case["kv"], case["head"], [place] * case["slots"])]
    at = _tensor(torch.tensor([[place]], dtype=torch.int32, device="cuda"))
    # a block of a stack: its input norm comes from the block before, its down product ends in the next block's norm
    h = llama.rms(xs, p["input_layernorm"], c).realize()
    s["keep"] = (p, xs, then, rot, at, h)
    s["rec"], s["out"] = _replayed(lambda: llama.slots_layer(xs, p, c, rot, keys, values, at, h=h, then=then))
    s["out"] += [_torch(keys), _torch(values)]
  elif kind == "block":
    c, p = _config(case, case["head"]), _upload_block(x["weights"], case["fmt"])
    places = np.arange(case["start"], case["start"] + case["tokens"], dtype=np.int32)
    rot = [_tensor(t) for t in _tables(case["heads"], case["kv"], case["head"], places)]
    rows = _tensor(torch.from_numpy(places[None]).cuda())
    s["block"] = (_tensor(x["x"]), p, c, rot, rows.reshape(1, case["tokens"], 1), _tensor(x["cache"]), rows)
    s["cache"] = _torch(s["block"][5])
  elif kind == "attend":
    rep = case["heads"] // case["kv"]
    cache = lambda t: (_tensor(t).cast(case["cache"]) if case["cache"] != "bf16" else _tensor(t)).realize().repeat_interleave(rep)
    s["calls"] = [(_tensor(q), cache(k), cache(v)) for q, k, v in zip(x["q"], x["k"], x["v"])]
    s["places"] = _tensor(x["places"])
    if case["rows"] == 1:
      s["rec"], s["out"] = _replayed(lambda: [q.attend(k, v, s["places"]) for q, k, v in s["calls"]])
  elif kind == "linear":
    s["x"], s["w"] = _tensor(x["x"]), [_columns(w, case["fmt"]) for w in x["w"]]
    s["r"] = _tensor(x["r"]) if case["act"] == "residual" else None
    if case["layers"] > 1:
      s["rec"], s["out"] = _replayed(lambda: [_linear(s, w).realize() for w in s["w"]])
  elif kind == "pack":
    s["w"] = _tensor(x["w"])
  else:
    s.update({k: _tensor(v) for k, v in x.items()})
  _runtime().wait()
  torch.cuda.synchronize()
  return s


def _linear(s, w):
  act, x = s["case"]["act"], s["x"]
  if act == "residual": return s["r"] + x.matmul(w, "fp32")
  y = x @ w
  return y.relu() if act == "relu" else y.silu() if act == "silu" else y


def run(s):
  case = s["case"]
  if "rec" in s:
    s["rec"].send()
    return s["out"]
  kind = case["kind"]
  if kind == "block": return [_torch(llama.layer(*s["block"])), s["cache"]]
  if kind == "attend":
    q, k, v = s["calls"][0]
    return _torch(q.attend(k, v, s["places"]))
  if kind == "linear": return _torch(_linear(s, s["w"][0]).realize())
  if kind == "pack": return _torch(s["w"].cast(case["fmt"]).columns().cast("bf16"))
  y = s["x"].layernorm() * s["w"] + s["b"] if case["op"] == "layernorm" else s["x"].softmax()
  return _torch(y.realize())


# ---- what a pass cannot do without

BYTES = {"bf16": 2.0, "bfp8": 17 / 16, "bfp4": 9 / 16}


def _block_work(case, hd, tokens, pairs, seen, fmt):
  """A block's bytes and flops for `tokens` rows: its matrices, `seen` cache rows read (over all sequences) and
  `pairs` query-key pairs a head."""
  q, kv = case["heads"] * hd, case["kv"] * hd
  values = case["dim"] * (q + 2 * kv) + q * case["dim"] + 3 * case["dim"] * case["ffn"]
  return {"bytes": values * BYTES[fmt] + seen * 2 * kv * 2 + tokens * 2 * kv * 2,
          "flops": 2 * tokens * values + 4 * pairs * q}


def work(case):
  kind = case["kind"]
  if kind == "step":
    hd, n = case["dim"] // case["heads"], max(1, case["slots"])
    seen = n * (case["at"] + 1) * (0.75 if case["slots"] else 1)  # places from half of `at` to `at`
    b = _block_work(case, hd, n, seen, seen, case["fmt"])
    head = case["dim"] * case["vocab"]
    return {"bytes": case["layers"] * b["bytes"] + head * BYTES[case["fmt"]] + n * (case["dim"] * 2 + case["vocab"] * 4),
            "flops": case["layers"] * b["flops"] + 2 * n * head}
  if kind == "slots":
    n = case["slots"]
    b = _block_work(case, case["head"], n, n * case["size"], n * case["size"], case["fmt"])
    return {"bytes": b["bytes"] + n * case["dim"] * (4 + 2 + 4 + 2), "flops": b["flops"]}
  if kind == "block":
    n = case["tokens"]
    b = _block_work(case, case["head"], n, n * case["start"] + n * (n + 1) / 2, case["start"], case["fmt"])
    return {"bytes": b["bytes"] + n * case["dim"] * 8, "flops": b["flops"]}
  if kind == "attend":
    n, r, keys = case["batch"], case["rows"], case["keys"]
    pairs = n * (r * (keys - r) + r * (r + 1) / 2) * (0.75 if case["ragged"] else 1)
    seen = n * keys * (0.75 if case["ragged"] else 1)
    return {"bytes": case["layers"] * (seen * 2 * case["kv"] * case["head"] * BYTES[case["cache"]] +
                                       4 * n * r * case["heads"] * case["head"]),
            "flops": case["layers"] * 4 * pairs * case["heads"] * case["head"]}
  if kind == "linear":
    m, k, n = case["m"], case["k"], case["n"]
    return {"bytes": 2 * m * k + case["layers"] * (k * n * BYTES[case["fmt"]] + m * n * (8 if case["act"] == "residual" else 2)),
            "flops": 2.0 * case["layers"] * m * k * n}
  size = case["rows"] * case["cols"]
  if kind == "pack":  # the source, its tiles written and read back, the values
    return {"bytes": size * (2 + 2 * BYTES[case["fmt"]] + 2), "flops": 0}
  return {"bytes": 2.0 * case["batch"] * size * (2 if case["dtype"] == "bf16" else 4), "flops": 0}


# ---- how far another correct implementation may be off: about four times what these paths are from 64 bits

def tolerance(case):
  kind = case["kind"]
  if kind == "pack": return "exact"
  if kind == "step": return {"rel": 1.5e-2, "max": 0.2}
  if kind in ("slots", "block"): return {"rel": 2e-2, "max": 0.2}
  if kind == "attend": return {"rel": 1e-2, "max": 0.1}
  if kind == "linear": return {"rel": 5e-6, "max": 5e-5} if case["act"] == "residual" else {"rel": 1e-2, "max": 5e-2}
  return {"rel": 5e-6, "max": 5e-5} if case["dtype"] == "fp32" else {"rel": 1.5e-2, "max": 0.1}


# ---- the same in 64 bits, in plain torch

def _block_float(w, fmt):
  """The values that the last axis's runs of 16 keep: 7 (bfp8) or 3 (bfp4) bits under the run's largest exponent."""
  if fmt == "bf16": return w.double()
  n = w.shape[-1]
  pad = torch.nn.functional.pad(w, (0, -n % 16)).reshape(*w.shape[:-1], -1, 16)
  bits = pad.view(torch.int16).to(torch.int32)
  e = bits >> 7 & 255
  m = (bits & 127) | (e != 0).to(torch.int32) << 7
  top = e.amax(-1, keepdim=True)
  shift = (top - e).clamp_(max=8)
  if fmt == "bfp8": q = ((m + (1 << shift)) >> (shift + 1)).clamp_(max=127)
  else: q = ((m + (16 << shift)) >> (shift + 5)).clamp_(max=7)
  q = torch.where(bits < 0, -q, q).double()
  return torch.ldexp(q, top - (133 if fmt == "bfp8" else 129)).reshape(*w.shape[:-1], -1)[..., :n]


def _attend64(q, k, v, lo, hi):
  """q (S, n, heads, hd), k and v (S, kv, keys, hd), the keys lo..hi of each row (S, n): (S, n, heads, hd)."""
  S, n, heads, hd = q.shape
  kv, keys = k.shape[1:3]
  rep, out = heads // kv, torch.empty_like(q)
  at = torch.arange(keys, device=q.device)
  hidden = (at < lo[..., None]) | (at > hi[..., None])
  for s in range(S):
    for g in range(kv):
      for r in range(0, n, 1024):
        part = q[s, r:r + 1024, g * rep:(g + 1) * rep]
        score = torch.matmul(part.transpose(0, 1), k[s, g].double().T)
        score.masked_fill_(hidden[s, r:r + 1024][None], -math.inf)
        out[s, r:r + 1024, g * rep:(g + 1) * rep] = torch.matmul(score.softmax(-1), v[s, g].double()).transpose(0, 1)
  return out


def _rms64(x, w): return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _block64(x, p, case, hd, places, k, v, rows, lo, fmt, h=None):
  """One block over x (S, n, dim); k and v (S, kv, size, hd) take the new rows at `rows` (S, n) and are read over each
  row's lo .. its own row. p's matrices are the stored values' sources."""
  S, n, _ = x.shape
  heads, kv = case["heads"], case["kv"]
  cos, sin = (t.view(S, n, heads + 2 * kv, hd).double() for t in _tables(heads, kv, hd, places))
  qkv = ((_rms64(x, p["input_layernorm"]) if h is None else h) @ _block_float(p["qkv_proj"], fmt)).view(S, n, heads + 2 * kv, hd)
  turned = torch.cat([-qkv[..., hd // 2:], qkv[..., :hd // 2]], -1)
  y = qkv * cos + turned * sin
  k, v = k.double(), v.double()
  for s in range(S):
    k[s][:, rows[s]], v[s][:, rows[s]] = y[s, :, heads:heads + kv].transpose(0, 1), y[s, :, heads + kv:].transpose(0, 1)
  o = _attend64(y[:, :, :heads].contiguous(), k, v, lo, rows)
  x = x + o.reshape(S, n, heads * hd) @ _block_float(p["o_proj"], fmt)
  gate_up = _rms64(x, p["post_attention_layernorm"]) @ _block_float(p["gate_up_proj"], fmt)
  gate, up = gate_up.chunk(2, -1)
  return x + (torch.nn.functional.silu(gate) * up) @ _block_float(p["down_proj"], fmt), k, v


def exact(case, seed):
  x, kind = _inputs(case, seed), case["kind"]
  if kind == "step":
    hd, kv, n = case["dim"] // case["heads"], case["kv"], max(1, case["slots"])
    places = x["places"].long()
    lo = torch.arange(n, device="cuda") * case["size"]
    y, caches = x["embed"][x["ids"].long()].double()[None], []
    for p, cache in zip(x["layers"], x["caches"]):
      y, k, v = _block64(y, p, case, hd, places.cpu().numpy(), cache[None, :kv], cache[None, kv:], (lo + places)[None], lo[None],
                         case["fmt"])
      caches.append(torch.cat([k[0], v[0]]))
    head = _block_float(x["embed"].T.contiguous(), case["fmt"])
    logits = _rms64(y, x["norm"]) @ head
    best = logits.max(-1, keepdim=True)
    return [logits] + ([best.values, None] if case["slots"] else []) + caches
  if kind == "slots":
    n, kv, size = case["slots"], case["kv"], case["size"]
    h = _rms64(x["x"].double(), x["weights"]["input_layernorm"])[:, None]
    rows = torch.full((n, 1), size - 1, device="cuda")
    shape = (n, kv, size, case["head"])
    y, k, v = _block64(x["x"].double()[:, None], x["weights"], case, case["head"], [size - 1] * n, x["keys"].view(shape),
                       x["values"].view(shape), rows, torch.zeros_like(rows), case["fmt"], h)
    return [y.view(1, n, -1), _rms64(y, x["then"]).view(1, n, -1), k.reshape(n * kv, size, -1), v.reshape(n * kv, size, -1)]
  if kind == "block":
    n, kv = case["tokens"], case["kv"]
    rows = torch.arange(case["start"], case["start"] + n, device="cuda")[None]
    y, k, v = _block64(x["x"].double()[None], x["weights"], case, case["head"], rows[0].cpu().numpy(), x["cache"][None, :kv],
                       x["cache"][None, kv:], rows, torch.zeros_like(rows), case["fmt"])
    return [y, torch.cat([k[0], v[0]])]
  if kind == "attend":
    b, heads, kv = case["batch"], case["heads"], case["kv"]
    hi = x["places"].view(b, heads, case["rows"])[:, 0].long()
    outs = []
    for q, k, v in zip(x["q"], x["k"], x["v"]):
      k, v = (_block_float(t, case["cache"]).view(b, kv, case["keys"], -1) for t in (k, v))
      q = q.double().view(b, heads, case["rows"], -1).transpose(1, 2).contiguous()
      o = _attend64(q, k, v, torch.zeros_like(hi), hi)
      outs.append(o.transpose(1, 2).reshape(b * heads, case["rows"], -1))
    return outs if case["rows"] == 1 else outs[0]
  if kind == "linear":
    outs = []
    for w in x["w"]:
      y = x["x"].double() @ _block_float(w, case["fmt"])
      outs.append(y.relu() if case["act"] == "relu" else torch.nn.functional.silu(y) if case["act"] == "silu" else
                  x["r"] + y if case["act"] == "residual" else y)
    outs = [y[None] for y in outs]
    return outs if case["layers"] > 1 else outs[0]
  if kind == "pack": return _block_float(x["w"], case["fmt"])[None]
  t = x["x"].double()
  if case["op"] == "softmax": return t.softmax(-1)
  t = t - t.mean(-1, keepdim=True)
  return t * torch.rsqrt((t * t).mean(-1, keepdim=True) + EPS) * x["w"].double() + x["b"].double()
