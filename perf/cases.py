"""What this framework is used for, as cases that can be timed and checked.

All but a few of the registry's published checkpoints run on one decoder (GQA
attention, SwiGLU or routed experts): these cases are its prompt passes, decode
steps and training passes, whole or as one stage of a ring. Sizes are those of
the registry's cards, of the serving defaults (8 slots of 4096 positions, prompt
chunks of 256 tokens) and of bench.py (128 sequences after prompts of 512).

  prefill  a prompt, or a chunk that follows `start` cached positions, eager
  decode   one token for every row, replayed from a captured graph as the ring
           and the serving worker do; `ragged` rows have their own lengths
  train    forward and backward of the cache-free pass: of a middle stage from a
           received gradient (`rank` > 0: of LoRA adapters), or of a last stage
           from the masked cross-entropy

Weights are random with the spread of a freshly initialised model, caches hold
random rows, norms lie around one.
"""
from __future__ import annotations

import math
import zlib

import torch

from xotorch_amd import ops
from xotorch_amd.engine.kvcache import make_cache
from xotorch_amd.models import model_class_for
from xotorch_amd.models.config import config_from_hf
from xotorch_amd.models.registry import builtin_config
from xotorch_amd.shard import Shard
from xotorch_amd.train.lora import apply_lora, lora_parameters

DEVICE = "cuda"
BF16 = torch.bfloat16


def listed():
  return [
    # one chat reply of a small model on one GPU: nothing but latency
    {"name": "decode-1b", "kind": "decode", "model": "llama-3.2-1b", "first": 0, "last": 15,
     "batch": 1, "context": 220, "capacity": 1024, "ragged": False},
    # the serving worker at its defaults: 8 slots, each as far as its own request is
    {"name": "decode-7b-slots", "kind": "decode", "model": "qwen-2.5-7b", "first": 0, "last": 27,
     "batch": 8, "context": 3100, "capacity": 4096, "ragged": True},
    # the headline benchmark's step on one of 8 GPUs: 128 sequences after a 512-token prompt
    {"name": "decode-70b-stage", "kind": "decode", "model": "llama-3-70b", "first": 30, "last": 39,
     "batch": 128, "context": 530, "capacity": 572, "ragged": False},
    # few long conversations on one of 4 GPUs: attention over the cache
    {"name": "decode-8b-long", "kind": "decode", "model": "llama-3-8b", "first": 8, "last": 15,
     "batch": 4, "context": 8000, "capacity": 8192, "ragged": True},
    # routed experts, one of 8 GPUs
    {"name": "decode-experts", "kind": "decode", "model": "mixtral-8x7b", "first": 8, "last": 11,
     "batch": 32, "context": 700, "capacity": 1024, "ragged": True},
    # a question of one line to a small model
    {"name": "prompt-1b-short", "kind": "prefill", "model": "llama-3.2-1b", "first": 0, "last": 15,
     "batch": 1, "seq": 45, "start": 0, "capacity": 557},
    # one chunk of a prompt that is served while other slots decode
    {"name": "prompt-7b-chunk", "kind": "prefill", "model": "qwen-2.5-7b", "first": 0, "last": 27,
     "batch": 1, "seq": 256, "start": 1280, "capacity": 4096},
    # a long document in one pass, first of 4 stages
    {"name": "prompt-8b-document", "kind": "prefill", "model": "llama-3-8b", "first": 0, "last": 7,
     "batch": 1, "seq": 6001, "start": 0, "capacity": 6513},
    # the headline benchmark's prompts on one of 8 GPUs
    {"name": "prompt-70b-stage", "kind": "prefill", "model": "llama-3-70b", "first": 30, "last": 39,
     "batch": 16, "seq": 512, "start": 0, "capacity": 572},
    # prompts through routed experts
    {"name": "prompt-experts", "kind": "prefill", "model": "mixtral-8x7b", "first": 8, "last": 11,
     "batch": 3, "seq": 700, "start": 0, "capacity": 1024},
    # fine-tuning of adapters, a middle one of 8 stages
    {"name": "train-adapters", "kind": "train", "model": "llama-3-8b", "first": 12, "last": 15,
     "batch": 8, "seq": 512, "rank": 8},
    # fine-tuning of all weights of a small model, the last of two stages
    {"name": "train-1b", "kind": "train", "model": "llama-3.2-1b", "first": 8, "last": 15,
     "batch": 2, "seq": 333, "rank": 0},
  ]


# model -> layers of one stage; the small ones whole
_STAGE = {"llama-3.2-1b": 16, "qwen-2.5-1.5b": 28, "qwen-2.5-7b": 28, "llama-3-8b": 8, "llama-3-70b": 10,
          "mixtral-8x7b": 4}


def _spread(rng, lo, hi):
  """A whole number between lo and hi, even over the logarithm."""
  return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
  kind = rng.choice(["decode", "decode", "prefill", "prefill", "train"])
  if kind == "train":
    if rng.random() < 0.5:
      seq = _spread(rng, 40, 1000)
      return {"kind": "train", "model": "llama-3-8b", "first": 12, "last": 15,
              "batch": _spread(rng, 1, max(1, min(8, 4096 // seq))), "seq": seq, "rank": rng.choice([4, 8, 16])}
    seq = _spread(rng, 40, 660)
    return {"kind": "train", "model": "llama-3.2-1b", "first": 8, "last": 15,
            "batch": _spread(rng, 1, max(1, min(4, 1320 // seq))), "seq": seq, "rank": 0}
  model = rng.choice(list(_STAGE))
  layers = _STAGE[model]
  total = builtin_config(model)["num_hidden_layers"]
  first = 0 if layers == total else rng.randrange(0, total - layers)
  case = {"kind": kind, "model": model, "first": first, "last": first + layers - 1}
  if kind == "decode":
    context = _spread(rng, 40, 8000)
    batch = _spread(rng, 1, max(1, min(128, 70000 // context)))
    ragged = batch > 1 and rng.random() < 0.6
    return {**case, "batch": batch, "context": context, "capacity": context + _spread(rng, 8, 190), "ragged": ragged}
  most = 8192 if model in ("llama-3-70b", "qwen-2.5-7b") else 12000
  seq = _spread(rng, 9, 6000)
  batch = 1 if rng.random() < 0.4 else _spread(rng, 1, max(1, min(64, most // seq)))
  if model == "mixtral-8x7b":
    batch = max(1, min(batch, 2100 // seq))
    seq = min(seq, 2100)
  start = 256 * rng.randrange(1, 9) if batch == 1 and seq <= 256 else 0
  return {**case, "batch": batch, "seq": seq, "start": start, "capacity": start + seq + _spread(rng, 8, 512)}


# ---------------- inputs ----------------

def _random(seed, name, shape, std, mean=0.0, dtype=BF16):
  """The values that go by `name`, whoever asks for them."""
  g = torch.Generator(device=DEVICE)
  g.manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
  return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(mean, std, generator=g)


def _whole(seed, name, shape, hi):
  g = torch.Generator(device=DEVICE)
  g.manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
  return torch.randint(0, hi, shape, generator=g, device=DEVICE)


def _stage(case):
  raw = builtin_config(case["model"])
  return raw, Shard(case["model"], case["first"], case["last"], raw["num_hidden_layers"])


def _head_dim(raw):
  return raw.get("head_dim") or raw["hidden_size"] // raw["num_attention_heads"]


def _spread_of(name, raw):
  """(std, mean) of a weight; what writes to the stream is the smaller the more layers do so."""
  if name.endswith("norm.weight"):
    return 0.1, 1.0
  if name.endswith("bias"):
    return 0.1, 0.0
  if name == "embed_tokens.weight":
    return 1.0, 0.0
  writes = name.endswith(("o_proj.weight", "down_proj.weight"))
  return 0.02 / (math.sqrt(2 * raw["num_hidden_layers"]) if writes else 1.0), 0.0


def _lengths(case, seed):
  """Cached positions of every row before this step."""
  n = case["context"]
  if not case["ragged"]:
    return [n] * case["batch"]
  part = _whole(seed, "lengths", (case["batch"],), max(1, n - n // 3)).tolist()
  return [n - p for p in part]


def _cached(case, seed, i, raw, rows):
  """Keys and values of `rows` earlier positions of local layer i: [B, rows, heads, dim]."""
  shape = (case["batch"], rows, raw["num_key_value_heads"], _head_dim(raw))
  return _random(seed, f"k{i}", shape, 1.3), _random(seed, f"v{i}", shape, 1.0)


def _inputs(case, seed, seq):
  raw, shard = _stage(case)
  if shard.is_first_layer:
    return _whole(seed, "tokens", (case["batch"], seq), raw["vocab_size"])
  # what earlier layers leave is several times what one of them adds
  return _random(seed, "hidden", (case["batch"], seq, raw["hidden_size"]), 3.0)


def _model(case, seed):
  raw, shard = _stage(case)
  cfg = config_from_hf(raw, case["model"])
  before = torch.get_default_dtype()
  torch.set_default_dtype(BF16)
  try:
    with torch.device("meta"):
      model = model_class_for(cfg)(cfg, shard)
  finally:
    torch.set_default_dtype(before)
  model = model.to_empty(device=DEVICE).to(BF16)
  model.reset_rope()
  with torch.no_grad():
    for name, p in model.named_parameters():
      p.copy_(_random(seed, name, p.shape, *_spread_of(name, raw)))
  return cfg, shard, model


def _fill(case, seed, raw, cache, rows):
  """Earlier positions into every layer's cache, as a prompt pass leaves them there."""
  heads, dim = raw["num_attention_heads"], _head_dim(raw)
  still, none = torch.ones(rows, dim // 2, device=DEVICE), torch.zeros(rows, dim // 2, device=DEVICE)
  at = torch.arange(rows, dtype=torch.int32, device=DEVICE)
  for i, layer in enumerate(cache.caches):
    k, v = _cached(case, seed, i, raw, rows)
    q = k.new_zeros(case["batch"], rows, heads, dim)
    qkv = torch.cat([q, k, v], dim=2).flatten(2)
    ops.rope_qkv_append(qkv, still, none, at, layer[0], layer[1], heads, raw["num_key_value_heads"], dim,
                        layer[2], layer[3])


def prepare(case, seed):
  raw, _ = _stage(case)
  cfg, shard, model = _model(case, seed)
  if case["kind"] == "train":
    model.train()
    if case["rank"]:
      apply_lora(model, rank=case["rank"], alpha=2.0 * case["rank"])
      with torch.no_grad():
        for name, p in model.named_parameters():
          if "lora_" in name:
            p.copy_(_random(seed, name, p.shape, 0.02, dtype=torch.float32))
    x = _inputs(case, seed, case["seq"]).requires_grad_(True)
    state = {"case": case, "model": model, "x": x, "params": [p for p in model.parameters() if p.requires_grad],
             "names": [n for n, p in model.named_parameters() if p.requires_grad],
             "positions": torch.arange(case["seq"], dtype=torch.int32, device=DEVICE)}
    if shard.is_last_layer:
      state["targets"] = _whole(seed, "targets", (case["batch"], case["seq"]), raw["vocab_size"])
      state["lengths"] = _whole(seed, "lengths", (case["batch"],), case["seq"] // 2) + (case["seq"] - case["seq"] // 2 + 1)
    else:
      state["gradient"] = _random(seed, "gradient", x.shape, 1.0)
    return state

  model.eval()
  cache = make_cache(cfg, shard, case["batch"], case["capacity"], BF16, DEVICE)
  state = {"case": case, "model": model, "caches": cache.caches}
  with torch.inference_mode():
    model.pack_decode_weights(reserve_bytes=24 << 30)
    if case["kind"] == "prefill":
      if case["start"]:
        _fill(case, seed, raw, cache, case["start"])
      state["x"] = _inputs(case, seed, case["seq"])
      state["positions"] = torch.arange(case["start"], case["start"] + case["seq"], dtype=torch.int32, device=DEVICE)
      return state
    _fill(case, seed, raw, cache, case["context"])
    lengths = _lengths(case, seed)
    x = _inputs(case, seed, 1)
    positions = torch.tensor(lengths if case["ragged"] else lengths[:1], dtype=torch.int32, device=DEVICE)
    seq_lens = torch.tensor(lengths, dtype=torch.int32, device=DEVICE) + 1

    def step():
      return model(x, caches=cache.caches, positions=positions, start_pos=-1, is_decode=True, seq_lens=seq_lens)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
      for _ in range(2):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
      state["out"] = step()
    state.update(graph=graph, held=(x, positions, seq_lens))
  return state


def run(state):
  case = state["case"]
  if case["kind"] == "train":
    for p in state["params"]:
      p.grad = None
    x = state["x"]
    x.grad = None
    out = state["model"](x, caches=None, positions=state["positions"], start_pos=0, last_only=False)
    if "targets" not in state:
      out.backward(state["gradient"])
      result = {"hidden": out.detach()}
    else:
      keep = torch.arange(case["seq"], device=x.device)[None, :] < state["lengths"][:, None]
      each = torch.nn.functional.cross_entropy(out.float().flatten(0, 1), state["targets"].flatten(), reduction="none")
      loss = (each.view(keep.shape) * keep).sum() / keep.sum().clamp(min=1)
      loss.backward()
      result = {"logits": out.detach(), "loss": loss.detach()}
    return {**result, "x": x.grad, "weights": {n: p.grad for n, p in zip(state["names"], state["params"])}}
  if case["kind"] == "decode":
    state["graph"].replay()
    out = state["out"]
  else:
    with torch.inference_mode():
      out = state["model"](state["x"], caches=state["caches"], positions=state["positions"], start_pos=case["start"])
  return {"out": out, "k": [c[0] for c in state["caches"]], "v": [c[1] for c in state["caches"]]}


# ---------------- what a pass cannot do without ----------------

def work(case):
  raw, shard = _stage(case)
  D, H, KVH, d = raw["hidden_size"], raw["num_attention_heads"], raw["num_key_value_heads"], _head_dim(raw)
  layers, B = shard.get_layer_count(), case["batch"]
  experts, top = raw.get("num_local_experts", 0), raw.get("num_experts_per_tok", 1)
  S = 1 if case["kind"] == "decode" else case["seq"]
  tokens = B * S
  attn, mlp = (H + 2 * KVH) * d * D + H * d * D, 3 * D * raw["intermediate_size"]
  head = raw["vocab_size"] * D if shard.is_last_layer else 0
  read = layers * (attn + mlp * (min(experts, tokens * top) if experts else 1)) + head
  used = layers * (attn + mlp * (top if experts else 1))
  ends = 2 * tokens * D * (1 if shard.is_first_layer else 2)
  if case["kind"] == "train":
    pairs = B * S * (S + 1) // 2
    dense = 2.0 * tokens * (used + head)
    flops = dense * (2 if case["rank"] else 3) + 3.5 * 4.0 * H * d * pairs * layers
    written = 0 if case["rank"] else 2 * read
    return {"bytes": 2.0 * read + written + 2 * ends, "flops": flops}
  if case["kind"] == "decode":
    pairs = sum(_expected(case)) + B
    rows = pairs + B
  else:
    pairs = B * (S * case["start"] + S * (S + 1) // 2)
    rows = B * (case["start"] + S)
  flops = 2.0 * tokens * used + 2.0 * B * head + 4.0 * H * d * pairs * layers
  return {"bytes": 2.0 * read + ends + 4.0 * rows * KVH * d * layers + 2 * B * (raw["vocab_size"] if head else 0), "flops": flops}


def _expected(case):
  n = case["context"]
  return [n] * case["batch"] if not case["ragged"] else [n - (n - n // 3) // 2] * case["batch"]


def tolerance(case):
  """Measured against 64 bits: up to 0.019 with 28 layers, 0.009 with few, 0.014 for gradients. A token
  whose second and third expert are as good as equal may go to either, which is seen in its row alone;
  norms' gradients are sums of many small terms."""
  loose = case["kind"] == "train" or "num_local_experts" in _stage(case)[0]
  return {"rel": 0.03, "max": 0.9 if loose else 0.4}


# ---------------- the same in 64 bits ----------------

def _norm64(x, w, eps):
  return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _angles64(raw, positions):
  """cos, sin [..., dim / 2] of positions."""
  dim = _head_dim(raw)
  freq = raw["rope_theta"] ** (-torch.arange(0, dim, 2, dtype=torch.float64, device=DEVICE) / dim)
  scaling = raw.get("rope_scaling")
  if scaling:
    wave = 2 * math.pi / freq
    old, lo, hi = scaling["original_max_position_embeddings"], scaling["low_freq_factor"], scaling["high_freq_factor"]
    part = ((old / wave - lo) / (hi - lo)).clamp(0, 1)
    freq = (1 - part) * freq / scaling["factor"] + part * freq
  angle = positions.double()[..., None] * freq
  return angle.cos(), angle.sin()


def _turn64(x, cos, sin):
  a, b = x.chunk(2, dim=-1)
  return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _attend64(q, k, v, last):
  """q [B,S,H,d], k and v [B,KVH,T,d]; query s of row b sees positions up to last[b,s]."""
  B, S, H, d = q.shape
  KVH = k.shape[1]
  rows = []
  for b in range(B):
    end = int(last[b].max()) + 1
    kb, vb = k[b, :, None, :end], v[b, :, None, :end]
    parts = []
    for s in range(0, S, 1024):
      qs = q[b, s:s + 1024].transpose(0, 1).reshape(KVH, H // KVH, -1, d)
      scores = qs @ kb.transpose(-1, -2) * d ** -0.5
      hidden = torch.arange(end, device=q.device)[None, :] > last[b, s:s + 1024, None]
      parts.append((scores.masked_fill(hidden, -math.inf).softmax(-1) @ vb).reshape(H, -1, d).transpose(0, 1))
    rows.append(torch.cat(parts).flatten(1))
  return torch.stack(rows)


def _swiglu64(x, gate_up, down):
  gate, up = (x @ gate_up.t()).chunk(2, dim=-1)
  return (torch.nn.functional.silu(gate) * up) @ down.t()


def _feed64(raw, weight, base, x):
  experts = raw.get("num_local_experts", 0)
  D, ff = raw["hidden_size"], raw["intermediate_size"]
  if not experts:
    return weight.apply(x, base + "mlp.gate_up_proj", (2 * ff, D), base + "mlp.down_proj", (D, ff))
  flat = x.flatten(0, 1)
  best, chosen = (flat @ weight(base + "mlp.gate.weight", (experts, D)).t()).softmax(-1).topk(raw["num_experts_per_tok"])
  best = best / best.sum(-1, keepdim=True)
  out = torch.zeros_like(flat)
  for e in range(experts):
    token, place = torch.where(chosen == e)
    if token.numel():
      name = f"{base}mlp.experts.{e}."
      y = _swiglu64(flat[token], weight(name + "gate_up_proj.weight", (2 * ff, D)), weight(name + "down_proj.weight", (D, ff)))
      out.index_add_(0, token, y * best[token, place, None])
  return out.view_as(x)


class _Weights:
  """Weights by name in 64 bits; the trained ones are leaves that are kept."""

  def __init__(self, case, seed):
    self.case, self.seed, self.raw, self.leaves = case, seed, _stage(case)[0], {}

  def __call__(self, name, shape):
    if self.case["kind"] != "train":
      return _random(self.seed, name, shape, *_spread_of(name, self.raw)).double()
    if "lora_" in name:
      self.leaves[name] = _random(self.seed, name, shape, 0.02, dtype=torch.float32).double().requires_grad_(True)
      return self.leaves[name]
    t = _random(self.seed, name, shape, *_spread_of(name, self.raw)).double()
    if not self.case["rank"]:
      self.leaves[name] = t.requires_grad_(True)
    return t

  def linear(self, x, name, shape, bias=False):
    y = x @ self(name + ".weight", shape).t()
    if bias:
      y = y + self(name + ".bias", (shape[0],))
    rank = self.case.get("rank", 0)
    if rank:
      y = y + 2.0 * (x @ self(name + ".lora_a", (rank, shape[1])).t()) @ self(name + ".lora_b", (shape[0], rank)).t()
    return y

  def apply(self, x, gate_up, wide, down, narrow):
    gate, up = self.linear(x, gate_up, wide).chunk(2, dim=-1)
    return self.linear(torch.nn.functional.silu(gate) * up, down, narrow)


def exact(case, seed):
  raw, shard = _stage(case)
  B, D, H, KVH, d = case["batch"], raw["hidden_size"], raw["num_attention_heads"], raw["num_key_value_heads"], _head_dim(raw)
  kind, bias, eps = case["kind"], raw["model_type"] == "qwen2", raw["rms_norm_eps"]
  weight = _Weights(case, seed)
  train = kind == "train"
  S = 1 if kind == "decode" else case["seq"]
  with torch.set_grad_enabled(train):
    x = _inputs(case, seed, S)
    if shard.is_first_layer:
      x = _random(seed, "embed_tokens.weight", (raw["vocab_size"], D), *_spread_of("embed_tokens.weight", raw))[x]
    x = x.double().requires_grad_(train)
    h = x
    if kind == "decode":
      before = _lengths(case, seed)
      at = torch.tensor(before, device=DEVICE)[:, None]
    else:
      at = (torch.arange(S, device=DEVICE) + case.get("start", 0)).expand(B, S)
    cos, sin = (t[:, :, None] for t in _angles64(raw, at))
    filled = case["context"] if kind == "decode" else case.get("start", 0)
    keys, values = [], []
    for i in range(shard.get_layer_count()):
      base = f"layers.{shard.start_layer + i}."
      qkv = weight.linear(_norm64(h, weight(base + "input_layernorm.weight", (D,)), eps), base + "self_attn.qkv_proj",
                          ((H + 2 * KVH) * d, D), bias)
      q, k, v = qkv.view(B, S, H + 2 * KVH, d).split([H, KVH, KVH], dim=2)
      q, k = _turn64(q, cos, sin), _turn64(k, cos, sin)
      if train:
        k_all, v_all = k.transpose(1, 2), v.transpose(1, 2)
      else:
        k_all, v_all = (torch.zeros(B, KVH, case["capacity"], d, dtype=torch.float64, device=DEVICE) for _ in range(2))
        if filled:
          old_k, old_v = _cached(case, seed, i, raw, filled)
          k_all[:, :, :filled], v_all[:, :, :filled] = old_k.transpose(1, 2).double(), old_v.transpose(1, 2).double()
        for b in range(B):
          k_all[b, :, at[b]], v_all[b, :, at[b]] = k[b].transpose(0, 1), v[b].transpose(0, 1)
        keys.append(k_all)
        values.append(v_all)
      mixed = _attend64(q, k_all, v_all, at)
      h = h + weight.linear(mixed, base + "self_attn.o_proj", (D, H * d))
      h = h + _feed64(raw, weight, base, _norm64(h, weight(base + "post_attention_layernorm.weight", (D,)), eps))
    if shard.is_last_layer:
      if not train:
        h = h[:, -1]
      h = _norm64(h, weight("norm.weight", (D,)), eps)
      head = "embed_tokens.weight" if shard.is_first_layer and raw.get("tie_word_embeddings") else "lm_head.weight"
      h = h @ weight(head, (raw["vocab_size"], D)).t()
    if not train:
      return {"out": h, "k": keys, "v": values}
    if shard.is_last_layer:
      targets = _whole(seed, "targets", (B, S), raw["vocab_size"])
      lengths = _whole(seed, "lengths", (B,), S // 2) + (S - S // 2 + 1)
      keep = torch.arange(S, device=DEVICE)[None, :] < lengths[:, None]
      each = torch.nn.functional.cross_entropy(h.flatten(0, 1), targets.flatten(), reduction="none")
      loss = (each.view(keep.shape) * keep).sum() / keep.sum().clamp(min=1)
      loss.backward()
      result = {"logits": h.detach(), "loss": loss.detach()}
    else:
      h.backward(_random(seed, "gradient", h.shape, 1.0).double())
      result = {"hidden": h.detach()}
    return {**result, "x": x.grad, "weights": {n: p.grad for n, p in weight.leaves.items()}}
