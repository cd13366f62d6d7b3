"""Whole stages of the GQA decoder on the GPU: what a layer fuses (products that a norm or an
attention kernel finishes, one or two rows with the norm inside) against 64 bits, beside
the same layers module by module; and modules that somebody watches."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
KINDS = {
  "tied": dict(n_heads=8, n_kv_heads=2, head_dim=64, tie_word_embeddings=True),
  "biased": dict(n_heads=6, n_kv_heads=2, head_dim=128, attn_bias=True),
  "normed": dict(n_heads=4, n_kv_heads=4, head_dim=128, qk_norm=True),
  "routed": dict(n_heads=4, n_kv_heads=1, head_dim=128, n_experts=4, n_experts_per_tok=2),
}
D, I, V, LAYERS = 512, 1024, 1000, 3


def _stage(kind, first, last, seed=0):
  from xotorch_amd.models.config import ModelConfig
  from xotorch_amd.models.llama import ShardedModel
  from xotorch_amd.shard import Shard
  cfg = ModelConfig(dim=D, intermediate_dim=I, vocab_size=V, n_layers=LAYERS, max_seq_len=512, rope_theta=10000.0, **KINDS[kind])
  model = ShardedModel(cfg, Shard("m", first, last, LAYERS)).cuda().to(BF).eval()
  g = torch.Generator(device="cuda").manual_seed(seed)
  with torch.no_grad():
    for name, p in model.named_parameters():
      std = 1.0 if "embed" in name else 0.1 if p.dim() == 1 else 0.3 if "gate.weight" in name else p.shape[-1] ** -0.5
      p.normal_(1.0 if "norm" in name else 0.0, std, generator=g)
  return cfg, model, g


def _norm(x, w, eps):
  return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


class Exact:
  """The stage in 64 bits: every call appends to the keys and values of each row."""

  def __init__(self, cfg, model):
    self.cfg, self.model, self.kv = cfg, model, [None] * len(model.layers)

  def __call__(self, x, at):
    """x [B, S] tokens or [B, S, D], at [B, S] positions -> stream or logits"""
    c, m = self.cfg, self.model
    h = m.embed_tokens.weight.double()[x] if x.dtype == torch.int64 else x.double()
    B, S = at.shape
    H, KVH, hd = c.n_heads, c.n_kv_heads, c.head_dim
    cos, sin = (torch.cat([t[at].double()] * 2, -1)[:, :, None] for t in (m.rope_cos, m.rope_sin))
    for i, layer in enumerate(m.layers.values()):
      a, mlp = layer.self_attn, layer.mlp
      y = _norm(h, layer.input_layernorm.weight, c.norm_eps) @ a.qkv_proj.weight.double().t()
      if c.attn_bias:
        y = y + a.qkv_proj.bias.double()
      q, k, v = y.view(B, S, H + 2 * KVH, hd).split([H, KVH, KVH], 2)
      if c.qk_norm:
        q, k = _norm(q, a.q_norm, c.norm_eps), _norm(k, a.k_norm, c.norm_eps)
      q, k = (t * cos + torch.cat([-t[..., hd // 2:], t[..., :hd // 2]], -1) * sin for t in (q, k))
      if self.kv[i] is None:
        self.kv[i] = [torch.zeros(B, 512, KVH, hd, dtype=torch.float64, device="cuda") for _ in "kv"]
      keys, values = self.kv[i]
      for b in range(B):
        keys[b, at[b]], values[b, at[b]] = k[b], v[b]
      end = int(at.max()) + 1
      kk, vv = (t[:, :end].repeat_interleave(H // KVH, 2).transpose(1, 2).contiguous() for t in (keys, values))
      s = q.transpose(1, 2) @ kk.transpose(-1, -2).contiguous() * hd ** -0.5
      s = s.masked_fill(torch.arange(end, device="cuda") > at[:, None, :, None], -torch.inf)
      h = h + (s.softmax(-1) @ vv).transpose(1, 2).flatten(2) @ a.o_proj.weight.double().t()
      y = _norm(h, layer.post_attention_layernorm.weight, c.norm_eps)
      if not c.n_experts:
        h = h + self._mlp(mlp, y)
      else:
        w, chosen = (y @ mlp.gate.weight.double().t()).softmax(-1).topk(c.n_experts_per_tok)
        w = w / w.sum(-1, keepdim=True)
        every = torch.stack([self._mlp(e, y) for e in mlp.experts], 2)
        h = h + (every.gather(2, chosen[..., None].expand(*chosen.shape, D)) * w[..., None]).sum(2)
    if m.shard.is_last_layer:
      h = _norm(h, m.norm.weight, c.norm_eps) @ m.head_weight().double().t()
    return h

  @staticmethod
  def _mlp(mlp, y):
    gate, up = (y @ mlp.gate_up_proj.weight.double().t()).chunk(2, -1)
    return (torch.nn.functional.silu(gate) * up) @ mlp.down_proj.weight.double().t()


def _input(model, B, S, g):
  if model.shard.is_first_layer:
    return torch.randint(0, V, (B, S), generator=g, device="cuda")
  return torch.randn(B, S, D, generator=g, device="cuda").to(BF) * 2


def _close(fast, apart, exact):
  """Rounded in the same places as module by module: no further from 64 bits, and every
  number within what some ten roundings to bf16 of a stream of this size add up to."""
  fast, apart = fast.double().view(exact.shape), apart.double().view(exact.shape)
  rows = exact.flatten(0, -2).norm(dim=-1).clamp(min=1e-9)
  off = [(t - exact).flatten(0, -2).norm(dim=-1) / rows for t in (fast, apart)]
  # a token whose experts are as good as equal may go to either: looked at by the median
  assert off[0].median() <= 1.2 * off[1].median() + 2.0 ** -10, (off[0].median(), off[1].median())
  assert off[0].quantile(0.97) <= 0.05
  size = exact.square().mean(-1, keepdim=True).sqrt()
  assert ((fast - exact).abs() > exact.abs() * 2.0 ** -6 + size * 0.2).double().mean() < 0.02


@pytest.mark.parametrize("kind,first,last", [("tied", 0, 2), ("tied", 1, 1), ("tied", 1, 2), ("biased", 0, 2), ("biased", 0, 1),
                                             ("normed", 1, 2), ("normed", 1, 1), ("routed", 0, 2), ("routed", 1, 2)])
@pytest.mark.parametrize("rows", [1, 2, 3, 17, 129, 256])
def test_a_stage_against_64_bits(kind, first, last, rows):
  from xotorch_amd.engine.kvcache import make_cache
  cfg, model, g = _stage(kind, first, last, seed=rows)
  B, S = rows, 5
  before = _input(model, B, S, g)
  steps = [(before, torch.arange(S, device="cuda").expand(B, S))]
  here = torch.randint(1, S + 1, (B,), generator=g, device="cuda")  # where each row goes on
  steps.append((_input(model, B, 1, g), here[:, None]))
  chunk = [(_input(model, 1, 4, g), torch.arange(4, device="cuda")[None]),
           (_input(model, 1, rows, g), torch.arange(4, 4 + rows, device="cuda")[None])]
  exact, found = Exact(cfg, model), []
  refs = [exact(*s) for s in steps]
  exact.kv = [None] * len(model.layers)
  refs += [exact(*s) for s in chunk]
  for watched in (False, True):
    hooks = [m.register_forward_hook(lambda *_: None) for m in model.modules()] if watched else []
    with torch.inference_mode():
      cache = make_cache(cfg, model.shard, B, 16, BF, "cuda")
      at = torch.arange(S, dtype=torch.int32, device="cuda")
      outs = [model(before, caches=cache.caches, positions=at, start_pos=0, last_only=False)]
      outs.append(model(steps[1][0], caches=cache.caches, positions=here.int(), start_pos=-1, is_decode=True,
                        seq_lens=here.int() + 1))
      cache = make_cache(cfg, model.shard, 1, rows + 4, BF, "cuda")
      for x, pos in chunk:
        outs.append(model(x, caches=cache.caches, positions=pos[0].int(), start_pos=int(pos[0, 0]), last_only=False))
    found.append([o.clone() for o in outs])
    for hook in hooks:
      hook.remove()
  for fast, apart, ref in zip(*found, refs):
    _close(fast, apart, ref)


@pytest.mark.parametrize("rows", [1, 3, 40, 200])
@pytest.mark.parametrize("kind", ["biased", "routed"])
def test_watched_modules_are_called(kind, rows):
  """A hook on a module of a stage sees its result, once a step, and can replace it. (The
  norm after attention is part of its residual sum, with a hook or without.)"""
  from xotorch_amd.engine.kvcache import make_cache
  cfg, model, g = _stage(kind, 0, 2)
  x = _input(model, rows, 1, g)
  at, seen = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.ones(rows, dtype=torch.int32, device="cuda")

  def step():
    with torch.inference_mode():
      cache = make_cache(cfg, model.shard, rows, 8, BF, "cuda")
      return model(x, caches=cache.caches, positions=at, start_pos=-1, is_decode=True, seq_lens=seen).float()

  plain = step()
  layer = model.layers["1"]
  watched = [layer, layer.input_layernorm, layer.self_attn, layer.self_attn.qkv_proj, layer.self_attn.o_proj,
             layer.mlp, model.norm, model.lm_head]
  watched += [layer.mlp.gate] if kind == "routed" else [layer.mlp.gate_up_proj, layer.mlp.down_proj]
  for module in watched:
    calls = []
    hook = module.register_forward_hook(lambda m, args, out: calls.append(out.shape))
    out = step()
    hook.remove()
    assert len(calls) == 1 and (out - plain).norm() <= 0.05 * plain.norm()
    hook = module.register_forward_hook(lambda m, args, out: -3 * out)
    assert (step() - plain).norm() > 0.1 * plain.norm()
    hook.remove()
    hook = module.register_forward_pre_hook(lambda m, args: calls.append(args[0].shape))
    step()
    hook.remove()
    assert len(calls) == 2
    forward = module.forward  # as libraries that move weights about do
    module.forward = lambda *args, **kw: (calls.append(None), forward(*args, **kw))[1]
    step()
    del module.forward
    assert len(calls) == 3


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("S,H,KVH,start,cap,window", [(1, 4, 2, 0, 30.0, 0), (45, 8, 2, 100, 0.0, 40), (130, 6, 1, 63, 20.0, 33),
                                                      (257, 4, 4, 1000, 0.0, 500), (70, 8, 8, 0, 10.0, 1)])
def test_prompt_attention_with_a_cap_or_a_window(hd, S, H, KVH, start, cap, window):
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  g = torch.Generator(device="cuda").manual_seed(S)
  c = ShardKVCache(1, 2, KVH, start + S, hd, BF, "cuda")[0]
  qkv = torch.randn(2, start + S, (H + 2 * KVH) * hd, generator=g, device="cuda").to(BF)
  still, none = torch.ones(start + S, hd // 2, device="cuda"), torch.zeros(start + S, hd // 2, device="cuda")
  ops.rope_qkv_append(qkv, still, none, torch.arange(start + S, dtype=torch.int32, device="cuda"), c.k, c.v, H, KVH, hd, c.kp, c.vp)
  q = qkv[:, start:, :H * hd].reshape(2, S, H, hd)
  scale = 0.2
  with torch.no_grad():
    out = ops.attn_prefill(q, c.k, c.v, start, S, c.kp, c.vp, scale=scale, softcap=cap, window=window).double()
  k, v = (t.double().repeat_interleave(H // KVH, 1) for t in (c.k, c.v))
  s = q.double().transpose(1, 2) @ k.transpose(-1, -2).contiguous() * scale
  if cap:
    s = cap * torch.tanh(s / cap)
  at, key = torch.arange(start, start + S, device="cuda")[:, None], torch.arange(start + S, device="cuda")[None]
  hidden = (key > at) | (key <= at - window) if window else key > at
  p = s.masked_fill(hidden, -torch.inf).softmax(-1)
  ref, size = (p @ v).transpose(1, 2), (p @ v.abs()).transpose(1, 2)
  # probabilities rounded to bf16 against the rounded sum; scores to fp32, tanh to some 2^-20 of the cap
  assert bool(((out - ref).abs() <= size * (2.0 ** -7 * 1.05 + cap * 2.0 ** -18) + ref.abs() * 2.0 ** -8 + 1e-6).all())
