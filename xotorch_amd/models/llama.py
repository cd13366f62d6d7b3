"""Sharded GQA transformer decoder for the llama / qwen2 / mistral families.

This is the framework's own decoder (capability parity with the reference's
torchtune assembly, /root/reference/xotorch/inference/torch/models/general_mha.py:23-254
and llm_utils.py:335-489), built for MI355X execution:

- every hot op goes through `xotorch_amd.ops` (HIP kernels on GPU, torch on CPU);
- KV caches are engine-owned, device-resident, laid out [B, KVH, T, hd] for
  the decode-attention kernel's row reads;
- a shard holds only layers [start_layer .. end_layer]; the first shard owns
  the token embedding, the last owns final norm + lm_head (tied embeddings
  supported);
- parameter names mirror HF checkpoints (q_proj/k_proj/... ) and RoPE uses
  the HF rotate-half convention, so safetensors load with no permute.
"""
from __future__ import annotations

import math
import os
from typing import Callable, List, Optional, Tuple

import torch
import torch.nn as nn

from xotorch_amd import ops
from xotorch_amd.models.config import ModelConfig
from xotorch_amd.ops import train_ops
from xotorch_amd.ops.torch_ref import rope_cos_sin
from xotorch_amd.shard import Shard


# (N, K, M) -> True when the packed skinny kernel beat hipBLASLt when timed
# in-situ (first eligible call at that M, before hipGraph capture).
_PACKED_WINS: dict = {}


def _time_us(fn, reps=4, rounds=3) -> float:
  """Min-of-rounds timing (DVFS / first-call noise makes a single round flip
  borderline auto-picks between runs)."""
  fn()  # warm
  best = float("inf")
  for _ in range(rounds):
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for _ in range(reps):
      fn()
    end.record()
    end.synchronize()
    best = min(best, start.elapsed_time(end) * 1000.0 / reps)
  return best


def _watched(*modules) -> bool:
  """Whether somebody waits for a call of one of these modules, whose work then is its own:
  a hook, or a forward that was put in place of the class's."""
  for m in modules:
    own = m.__dict__
    if own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own:
      return True
  return torch.nn.modules.module._has_any_global_hook()


def _own(module, name: str = "weight"):
  """module.weight (or another parameter) without nn.Module's search for it, which a pass
  through a small model makes some 700 times, a quarter of a microsecond each."""
  held = module._parameters
  return held[name] if name in held else getattr(module, name)


def _fastest(key, captured: str, **ways: Callable) -> str:
  """The fastest of these ways, timed now and kept in _PACKED_WINS. Any but the first has
  to win by 5%: closer ones would change from run to run. While a graph is captured
  nothing can be timed: `captured`."""
  if torch.cuda.is_current_stream_capturing():
    return captured
  times = {name: _time_us(f) for name, f in ways.items()}
  first = next(iter(ways))
  use = _PACKED_WINS[key] = min(times, key=lambda name: times[name] * (0.95 if name == first else 1.0))
  if os.getenv("XOT_DEBUG", "0") != "0":
    print(f"[xot] auto-pick {key}: " + ", ".join(f"{n} {t:.1f} us" for n, t in times.items()) + f" -> {use}", flush=True)
  return use


class XotLinear(nn.Linear):
  """nn.Linear whose bf16 inference products of up to 256 rows go by the kernels of
  hip/rows_ops.hip (up to ops.FEW_ROWS rows) and hip/tile_ops.hip (ops.tile_wins), which
  read the weight as it lies. `pack_decode()` stores a second copy in MFMA A-fragment
  order ([N/32,K/16,64,8], see ops.pack_decode_weight); with 32, 64 .. 256 rows these
  ways, the weight-streaming kernels that read the copy and hipBLASLt are timed at the
  first call and the fastest is kept (lm_head of 70B, 64 rows: 0.87 of the library's time
  by the copy, 1.07 by tiles). More rows and training go by ops.linear: the kernels of
  hip/gemm_ops.hip where train_ops.forward_wins, input_wins and weight_wins say so, else
  hipBLASLt; MLP.whole_gate takes gate and up of prompts in one kernel, past this
  forward. The CPU stays on aten. Storage and state dict are nn.Linear's."""

  hip = ("_hip_rows", "_hip_tile", "_hip_gemm")  # what a pass loads beside the operators
  weight_packed: Optional[torch.Tensor]

  def __init__(self, *a, **kw):
    super().__init__(*a, **kw)
    self.weight_packed = None
    self.weight_packed_fp8 = None
    self.weight_scale = None

  def packable(self) -> bool:
    N, K = self.weight.shape
    return N % 128 == 0 and K % 64 == 0

  def pack_decode(self):
    if self.packable() and self.weight.is_cuda and self.weight.dtype == torch.bfloat16:
      if ops.fp8_gemm_enabled():
        if getattr(self, "weight_packed_fp8", None) is None:
          self.weight_packed_fp8, self.weight_scale = ops.pack_decode_weight_fp8(self.weight.detach())
      elif self.weight_packed is None:
        self.weight_packed = ops.pack_decode_weight(self.weight.detach())

  def copied(self, rows: int) -> bool:
    """Whether a product of so many rows can read the packed copy."""
    return self.weight_packed is not None and 32 <= rows <= 256 and rows % 32 == 0

  def unpack_decode(self):
    self.weight_packed = None
    self.weight_packed_fp8 = None

  _w8 = None
  _w8_scale = None

  def _fp8_prefill(self, x):
    """Opt-in (XOT_FP8_PREFILL=1) e4m3 prefill GEMM via hipBLASLt scaled_mm:
    measured 2.58 vs 1.58 PF on the 70B gate_up prefill shape (rel err
    ~3.5%). Per-token activation scales, per-channel weight scales; the
    fp8 weight copy is cached lazily."""
    N, K = self.weight.shape
    M = x.numel() // K
    w8, sw = self._w8, self._w8_scale
    if w8 is None:
      w = self.weight.detach()
      sw = (w.float().abs().amax(dim=1, keepdim=True).clamp(min=1e-12) / 448.0)
      w8 = (w / sw.to(w.dtype)).clamp(-448, 448).to(torch.float8_e4m3fn)
      free, _ = torch.cuda.mem_get_info()
      if free > (12 << 30):  # persist the fp8 copy only with HBM headroom
        self._w8, self._w8_scale = w8, sw
    # activation quantization stays in bf16 (a fp32 image of a 65k x 8k
    # prefill activation would be 2 GB per layer)
    x2 = x.reshape(M, K)
    sx = (x2.abs().amax(dim=1, keepdim=True).float().clamp(min=1e-12) / 448.0)
    x8 = (x2 / sx.to(x2.dtype)).clamp(-448, 448).to(torch.float8_e4m3fn)
    y = torch._scaled_mm(x8, w8.t(), scale_a=sx, scale_b=sw.t(),
                         out_dtype=torch.bfloat16)
    if self.bias is not None:
      y = y + self.bias
    return y.view(list(x.shape[:-1]) + [N])

  def forward(self, x):
    if (x.is_cuda and x.dtype == torch.bfloat16 and not torch.is_grad_enabled()
        and os.getenv("XOT_FP8_PREFILL", "0") == "1"):
      N, K = self.weight.shape
      M = x.numel() // K
      if M > 256 and N % 16 == 0 and K % 16 == 0 and x.is_contiguous():
        try:
          return self._fp8_prefill(x)
        except torch.cuda.OutOfMemoryError:
          torch.cuda.empty_cache()  # fall back to the bf16 path
    wp8 = getattr(self, "weight_packed_fp8", None)
    if wp8 is not None and x.is_cuda and x.dtype == torch.bfloat16 and not torch.is_grad_enabled():
      N, K = self.weight.shape
      M = x.numel() // K
      if 32 <= M <= 256 and M % 32 == 0 and x.is_contiguous():
        from xotorch_amd.ops import _load_hip
        hip = _load_hip()
        if hip is not None:
          x8, sx = hip.quant_fp8_rows(x.view(M, K))
          y = hip.skinny_gemm_fp8(x8, sx, wp8, self.weight_scale, 1, N, self.bias)
          sizes = list(x.shape[:-1]) + [N]
          return y.view(sizes)
    if x.numel() <= ops.FEW_ROWS * self.in_features and ops.few_rows(x, self.weight) and (self.bias is None or self.bias.dtype == torch.bfloat16):
      return ops.rows_linear(x, self.weight, self.bias)
    if x.numel() <= ops.TILE_ROWS * self.in_features and ops.tile_rows(x, self.weight) and (self.bias is None or self.bias.dtype == torch.bfloat16):
      w, b = self.weight, self.bias
      N, K = w.shape
      M = x.numel() // K
      use = "tile" if ops.tile_wins(M, N, K) else "blaslt"
      if self.copied(M):
        from xotorch_amd.ops import _load_hip
        hip, wp = _load_hip(), self.weight_packed
        use = _PACKED_WINS.get((N, K, M)) or _fastest(
          (N, K, M), use if use == "tile" else "packed",
          blaslt=lambda: torch.nn.functional.linear(x, w, b), tile=lambda: ops.tile_linear(x, w, b),
          packed=lambda: hip.skinny_gemm_packed(x, wp, N, b), xreg=lambda: hip.skinny_gemm_packed_xreg(x, wp, N, b))
        if use == "xreg":
          return hip.skinny_gemm_packed_xreg(x, wp, N, b)
        if use == "packed":
          return hip.skinny_gemm_packed(x, wp, N, b)
      if use == "tile":
        return ops.tile_linear(x, w, b)
    return ops.linear(x, self.weight, self.bias)


class RMSNorm(nn.Module):
  def __init__(self, dim: int, eps: float):
    super().__init__()
    self.weight = nn.Parameter(torch.ones(dim))
    self.eps = eps

  def forward(self, x):
    return ops.rmsnorm(x, self.weight, self.eps)


class Attention(nn.Module):
  """GQA attention with a FUSED qkv projection: one [D, (H+2KVH)*hd] GEMM per
  layer instead of three (decode on MI355X is GEMM-launch bound at small
  batch); the packed output feeds the fused RoPE+KV-append kernel directly."""

  def __init__(self, cfg: ModelConfig):
    super().__init__()
    self.cfg = cfg
    H, KVH, hd, D = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim, cfg.dim
    self.qkv_proj = XotLinear(D, (H + 2 * KVH) * hd, bias=cfg.attn_bias)
    self.o_proj = XotLinear(H * hd, D, bias=False)
    if cfg.qk_norm:  # qwen3: per-head RMSNorm on q/k before RoPE
      self.q_norm = nn.Parameter(torch.ones(hd))
      self.k_norm = nn.Parameter(torch.ones(hd))

  def _forward_nocache(self, x, cos, sin, positions):
    """Cache-free causal attention (training/eval): the SAME modules and
    weights as the inference path, autograd-safe ops (fp32 sdpa). This is
    the one and only training forward — the engine calls the model, so the
    two paths cannot drift."""
    import torch.nn.functional as F
    B, S, _ = x.shape
    cfg = self.cfg
    H, KVH, hd = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim
    qkv = self.qkv_proj(x)
    if not cfg.qk_norm and train_ops.takes_heads(qkv, cos, sin, positions, hd):
      return self.o_proj(train_ops.causal_heads(qkv, cos, sin, positions, H, KVH, hd))
    q, k, v = torch.split(qkv, [H * hd, KVH * hd, KVH * hd], dim=-1)
    q = q.reshape(B, S, H, hd)
    k = k.reshape(B, S, KVH, hd)
    v = v.reshape(B, S, KVH, hd)
    if cfg.qk_norm:
      from xotorch_amd.ops import torch_ref as tr
      q = tr.rmsnorm(q.float(), self.q_norm.float(), cfg.norm_eps).to(q.dtype)
      k = tr.rmsnorm(k.float(), self.k_norm.float(), cfg.norm_eps).to(k.dtype)
    q, k = ops.rope_apply(q, k, cos, sin, positions)
    rep = H // KVH
    out = F.scaled_dot_product_attention(
      q.transpose(1, 2).float(),
      k.transpose(1, 2).repeat_interleave(rep, dim=1).float(),
      v.transpose(1, 2).repeat_interleave(rep, dim=1).float(),
      is_causal=True,
    ).to(x.dtype)
    return self.o_proj(out.transpose(1, 2).reshape(B, S, H * hd))

  def forward(self, x, cos, sin, positions, kv, start_pos: int, is_decode: bool, seq_lens=None):
    if kv is None:
      return self._forward_nocache(x, cos, sin, positions)
    qkv = self.qkv_proj(x)  # [B, S, (H+2KVH)*hd]
    return self.o_proj(self.attend(qkv, cos, sin, positions, kv, start_pos, is_decode, seq_lens))

  def project(self, x):
    """qkv_proj by weight tiles; where k is split, (a place for the queries, the sums over
    parts of k) for attend, whose first kernel adds them up."""
    p = self._modules["qkv_proj"]
    w = _own(p)
    if type(self) is Attention and ops.tile_parted(w, _own(p, "bias")):
      return x.new_empty(*x.shape[:-1], w.shape[0]), ops.tile_parts(x, w)
    return p(x), None

  def attend(self, qkv, cos, sin, positions, kv, start_pos: int, is_decode: bool, seq_lens=None, sums=None):
    """What lies between the projections: qkv [B, S, (H+2KVH)*hd] -> [B, S, H*hd]."""
    B, S, _ = qkv.shape
    cfg = self.cfg
    H, hd = cfg.n_heads, cfg.head_dim
    k_cache, v_cache = kv[0], kv[1]
    kp = kv[2] if len(kv) > 2 else None  # MFMA-packed cache copies (GPU, hd 64 or 128)
    vp = kv[3] if len(kv) > 3 else None
    ksc = kv[4] if len(kv) > 4 else None  # fp8-KV mode scales
    vsc = kv[5] if len(kv) > 5 else None
    qn = self.q_norm if cfg.qk_norm else None
    kn = self.k_norm if cfg.qk_norm else None
    bias = _own(self._modules["qkv_proj"], "bias") if sums is not None else None
    if is_decode and ops.decode_attends(qkv, H, cfg.n_kv_heads, hd, kp, qn, kn):
      sl = seq_lens if seq_lens is not None else start_pos + 1
      return ops.decode_attend(qkv, cos, sin, positions, sl, k_cache, v_cache, kp, vp, H, cfg.n_kv_heads,
                               qn, kn, cfg.norm_eps, sums, bias)
    ops.rope_qkv_append(qkv, cos, sin, positions, k_cache, v_cache, H, cfg.n_kv_heads, hd, kp, vp,
                        qn, kn, cfg.norm_eps, ksc, vsc, sums, bias)
    q = qkv[:, :, : H * hd].view(B, S, H, hd)  # strided view; kernels accept it
    if is_decode:
      sl = seq_lens if seq_lens is not None else start_pos + 1
      out = ops.attn_decode(q, k_cache, v_cache, sl, kp, vp, k_scale=ksc, v_scale=vsc)
    else:
      out = ops.attn_prefill(q, k_cache, v_cache, start_pos, S, kp, vp)
    return out.reshape(B, S, H * hd)


class MLP(nn.Module):
  """SwiGLU MLP with a FUSED gate+up projection ([D, 2I] GEMM); the packed
  [gate | up] output feeds the packed SwiGLU kernel."""

  def __init__(self, cfg: ModelConfig, intermediate: Optional[int] = None):
    super().__init__()
    I = intermediate or cfg.intermediate_dim
    self.intermediate = I
    self.gate_up_proj = XotLinear(cfg.dim, 2 * I, bias=False)
    self.down_proj = XotLinear(I, cfg.dim, bias=False)

  @staticmethod
  def act(gu):
    return ops.swiglu_packed(gu)

  def by_tiles(self, x) -> bool:
    """Whether gated() and parts of the down projection are this MLP."""
    gu, dp = self._modules["gate_up_proj"], self._modules["down_proj"]
    if type(gu) is not XotLinear or type(dp) is not XotLinear or _watched(self, gu, dp):
      return False
    up, down, rows = _own(gu), _own(dp), x.numel() // x.shape[-1]
    return (_own(gu, "bias") is None and _own(dp, "bias") is None
            and gu.weight_packed_fp8 is None and dp.weight_packed_fp8 is None
            and up.shape[0] % 8 == 0 and ops.tiled(x, up, down)
            and ops.parts_win(rows, *down.shape) and not dp.copied(rows))

  def gate_is_tile(self, x) -> bool:
    """Whether gated() is tile_swiglu without timing it."""
    gu = self._modules["gate_up_proj"]
    N, K = _own(gu).shape
    rows = x.numel() // K
    return ops.gate_wins(rows, N, K) and not gu.copied(rows)

  def gated(self, x):
    """The gated activation of x (by_tiles)."""
    gu = self.gate_up_proj
    N, K = gu.weight.shape
    rows = x.numel() // K
    tile = ops.gate_wins(rows, N, K)
    if tile and gu.copied(rows):
      key = "gate", N, K, rows
      tile = (_PACKED_WINS.get(key) or _fastest(key, "tile", tile=lambda: ops.tile_swiglu(x, gu.weight),
                                                split=lambda: self.act(gu(x)))) == "tile"
    return ops.tile_swiglu(x, gu.weight) if tile else self.act(gu(x))

  def whole_gate(self, x) -> bool:
    """Whether the gated activation of a prompt is one kernel (train_ops.takes_gate)."""
    # said first, as a pass through many experts asks some hundred times: 300 tokens through
    # two layers of 128 took 10.1 ms with all questions, 9.9 so
    if x.numel() <= 256 * x.shape[-1]:
      return False
    gu = self._modules["gate_up_proj"]
    return (type(self) is MLP and type(gu) is XotLinear and not _watched(gu) and _own(gu, "bias") is None
            and train_ops.takes_gate(x, _own(gu)) and os.getenv("XOT_FP8_PREFILL", "0") != "1")

  def forward(self, x):
    if self.whole_gate(x):
      return self.down_proj(train_ops.gate_product(x, self.gate_up_proj.weight))
    gu = self.gate_up_proj(x)
    dp = self.down_proj
    if (getattr(dp, "weight_packed", None) is not None and gu.is_cuda and gu.dtype == torch.bfloat16
        and not torch.is_grad_enabled() and gu.is_contiguous()
        and os.getenv("XOT_FUSE_SWIGLU", "1") == "1"):
      I = self.intermediate
      M = gu.numel() // (2 * I)
      if 32 <= M <= 256 and M % 32 == 0:
        from xotorch_amd.ops import _load_hip
        hip = _load_hip()
        if hip is not None:
          N = dp.weight.shape[0]
          key = ("fuse_swiglu", N, I, M)
          use = _PACKED_WINS.get(key)
          if use is None:
            if torch.cuda.is_current_stream_capturing():
              use = "fused"
            else:
              wp = dp.weight_packed
              t_fused = _time_us(lambda: hip.skinny_gemm_packed_swiglu(gu, wp, N, dp.bias))
              t_split = _time_us(lambda: dp(self.act(gu)))
              use = "fused" if t_fused < t_split * 0.98 else "split"
              _PACKED_WINS[key] = use
              if os.getenv("XOT_DEBUG", "0") != "0":
                print(f"[xot] swiglu-fuse auto-pick N={N} I={I} M={M}: fused {t_fused:.1f} us "
                      f"vs split {t_split:.1f} us -> {use}", flush=True)
          if use == "fused":
            y = hip.skinny_gemm_packed_swiglu(gu, dp.weight_packed, N, dp.bias)
            return y.view(list(x.shape[:-1]) + [N])
    return self.down_proj(self.act(gu))


class MoEMLP(nn.Module):
  """Mixtral-class sparse MoE block (top-k routed SwiGLU experts).

  bf16 inference on the GPU runs as grouped products that read tokens and weights
  where they lie (`_grouped`); shapes are static and the host sees no count, so that
  a graph can hold them. Else decode (<=256 tokens) runs a static-shape routed path:
  assignments are argsorted by expert, every expert
  gets a fixed token capacity C = round_up(T, 32) (top-k experts are distinct
  per token so a single expert can receive at most T assignments — lossless),
  padded slots carry weight 0, and the per-expert GEMMs run as ONE grouped
  MFMA launch on stacked prepacked weights (`skinny_gemm_grouped`) when
  packed, else per-expert XotLinear. Prefill/CPU/training use the dynamic
  gather loop (the reference's semantics, llm_utils.py:502-590)."""

  def __init__(self, cfg: ModelConfig):
    super().__init__()
    self.n_experts = cfg.n_experts
    self.top_k = cfg.n_experts_per_tok
    self.dim = cfg.dim
    self.intermediate = cfg.moe_intermediate_dim or cfg.intermediate_dim
    self.gate = nn.Linear(cfg.dim, cfg.n_experts, bias=False)
    self.experts = nn.ModuleList(
      [MLP(cfg, intermediate=self.intermediate) for _ in range(cfg.n_experts)]
    )
    self.wp_gate_up: Optional[torch.Tensor] = None
    self.wp_down: Optional[torch.Tensor] = None
    self.wp_gate_up_fp8: Optional[torch.Tensor] = None
    self.wp_down_fp8: Optional[torch.Tensor] = None
    self.sw_gate_up: Optional[torch.Tensor] = None
    self.sw_down: Optional[torch.Tensor] = None

  def pack_grouped(self):
    """Stack the experts' prepacked weights for the grouped decode GEMM."""
    if ops.fp8_gemm_enabled():
      if self.wp_gate_up_fp8 is None \
         and all(getattr(e.gate_up_proj, "weight_packed_fp8", None) is not None for e in self.experts) \
         and all(getattr(e.down_proj, "weight_packed_fp8", None) is not None for e in self.experts):
        self.wp_gate_up_fp8 = torch.stack([e.gate_up_proj.weight_packed_fp8 for e in self.experts]).contiguous()
        self.sw_gate_up = torch.stack([e.gate_up_proj.weight_scale for e in self.experts]).contiguous()
        self.wp_down_fp8 = torch.stack([e.down_proj.weight_packed_fp8 for e in self.experts]).contiguous()
        self.sw_down = torch.stack([e.down_proj.weight_scale for e in self.experts]).contiguous()
        for e in self.experts:
          e.gate_up_proj.weight_packed_fp8 = None
          e.down_proj.weight_packed_fp8 = None
      return
    if self.wp_gate_up is None and all(e.gate_up_proj.weight_packed is not None for e in self.experts) \
       and all(e.down_proj.weight_packed is not None for e in self.experts):
      self.wp_gate_up = torch.stack([e.gate_up_proj.weight_packed for e in self.experts]).contiguous()
      self.wp_down = torch.stack([e.down_proj.weight_packed for e in self.experts]).contiguous()
      for e in self.experts:  # the grouped stack supersedes the per-expert packs
        e.gate_up_proj.weight_packed = None
        e.down_proj.weight_packed = None

  def _route(self, flat):
    """Top-k routing -> normalized weights [T, k] + expert ids [T, k]."""
    router = self.gate(flat).float()
    weights, selected = torch.topk(torch.softmax(router, dim=-1), self.top_k, dim=-1)
    weights = weights / weights.sum(dim=-1, keepdim=True)
    return weights, selected

  def forward(self, x):
    B, S, D = x.shape
    flat = x.view(-1, D)
    T = flat.shape[0]
    if x.is_cuda and not torch.is_grad_enabled() and T <= 256:
      return self._forward_decode(flat).view(B, S, D).to(x.dtype)
    # NOTE: chunking the static grouped path over 256-token slices for
    # prefill was measured 1.5-2.5x WORSE TTFT (every chunk re-streams the
    # full expert weights; the eager loop streams each expert once with a
    # large-M GEMM). Instead, prefill sorts the token-expert pairs ONCE and
    # runs each expert on a contiguous slice — one argsort + one gather
    # replaces E per-expert where/eq scans over the full assignment list.
    if x.is_cuda and not torch.is_grad_enabled():
      found = self._grouped(flat)
      if found is not None:
        return self._forward_grouped(flat, found).view(B, S, D)
    weights, selected = self._route(flat)
    if x.is_cuda and not torch.is_grad_enabled():
      return self._forward_prefill_sorted(flat, weights, selected).view(B, S, D).to(x.dtype)
    out = torch.zeros_like(flat, dtype=torch.float32)
    for e in range(self.n_experts):
      token_idx, k_idx = torch.where(selected == e)
      if token_idx.numel() == 0:
        continue
      expert_out = self.experts[e](flat[token_idx]).float()
      out.index_add_(0, token_idx, expert_out * weights[token_idx, k_idx, None])
    return out.view(B, S, D).to(x.dtype)

  def _many(self, flat) -> bool:
    """Whether the grouped products go by tiles of 128 and 256 tokens: over 24 rows
    per expert (fewer leave most of a tile of 128 tokens empty), up to 256 tokens over 48: 8 experts
    of 4096 x 14336, two of them a token, us by tiles of up to 64 rows and by these: 128 tokens 460, 508;
    192 467, 516; 256 738, 563."""
    return flat.shape[0] * self.top_k > (24 if flat.shape[0] > 256 else 48) * self.n_experts

  def _expert_weights(self):
    """The experts' weights (gate and up of all, down of all) where grouped products may read them:
    bf16, one tensor per expert and projection, whose modules nobody waits for by a hook of their own. Else None.
    Straight from where modules keep things, as a pass through 128 experts asks 256 modules in
    every layer: 740 us by their attributes, 117 so (40 with 8 experts)."""
    if self.n_experts > 256 or self.top_k > 8 or self.dim % 64 or self.intermediate % 64 or max(self.dim, self.intermediate) > 1 << 22:
      return None
    ups, downs = [], []
    for e in self._modules["experts"]._modules.values():
      own = e.__dict__
      if type(e) is not MLP or own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own:
        return None
      held = own["_modules"]
      for p, found in ((held["gate_up_proj"], ups), (held["down_proj"], downs)):
        own = p.__dict__
        if type(p) is not XotLinear or own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own:
          return None
        params = own["_parameters"]
        if params.get("bias") is not None or params.get("weight") is None:
          return None
        found.append(params["weight"])
    return ups, downs

  def _grouped(self, flat):
    """The experts' weights where tokens go through them as two grouped products, and the router's where
    its logits are made with the choice; or None. Up to 256 tokens a router that somebody waits for, by a hook of
    its own or a global one, that is another module or has a bias, or that autocast or a dispatch mode takes, has its own
    call and the experts none: us of a layer with 1 and 32 tokens, expert by expert and so, 8 experts of 4096 x 14336 580, 155 and
    570, 444; 128 of 2048 x 768 4510, 148 and 4535, 203. More tokens go by the modules then."""
    few = flat.shape[0] <= 256
    if flat.dtype != torch.bfloat16 or not flat.is_cuda or not flat.is_contiguous() or not flat.numel():
      return None
    # fp8 copies are read up to 256 tokens, fp8 products of prompts are the modules'
    if self.wp_gate_up_fp8 is not None if few else os.getenv("XOT_FP8_PREFILL", "0") == "1":
      return None
    found = self._expert_weights()
    if found is None:
      return None
    gate = self._modules["gate"]
    alone = type(gate) is nn.Linear and _own(gate, "bias") is None and not _watched(gate) and ops.alone(flat)
    if not alone and (not few or train_ops.followed() or type(flat) not in train_ops.OWN):
      return None
    weights = [*found[0], *found[1]]
    if not ops._use_hip(flat) or flat.get_device() != train_ops._current_device() or any(type(w) not in train_ops.OWN for w in weights):
      return None
    from xotorch_amd.ops.mixer_ops import load_hip
    readable = load_hip("_hip_experts").readable
    router = _own(gate) if alone else None
    if alone and not (type(router) in train_ops.OWN and readable(flat, [router])):
      if not few:
        return None
      router = None
    return (*found, router) if readable(flat, weights) else None

  def _forward_grouped(self, flat, found, wide=False):
    """Rows of all (token, expert) pairs are placed by counting, without the host; the
    products read tokens and weights where they lie, of experts that have a row. `wide`: fp32."""
    from xotorch_amd.ops.mixer_ops import load_hip
    hip = load_hip("_hip_experts")
    ups, downs, router = found
    # tiles of 256 tokens from 110 rows an expert on: 8 experts of 4096 x 14336, two of
    # them a token, us with 128 and 256: 300 tokens 565, 577; 450 607, 602; 620 667, 578
    tile = 256 if flat.shape[0] * self.top_k >= 110 * self.n_experts else 128
    rule = None, self.top_k, 1, 1, 1.0, True, 0, False, False, tile
    if router is not None:
      # up to 256 tokens logits are rounded as those of the gate's own call, which hooks bring about
      weight, row, *places = hip.route(flat, router, *rule, flat.shape[0] <= 256)
    else:
      logits = self.gate(flat)
      weight, row, *places = hip.route((logits if logits.dtype == torch.bfloat16 else logits.float()).contiguous(), None, *rule)
    product = hip.expert_product_of if self._many(flat) else hip.expert_few_of
    y = product(product(flat, ups, *places, True), downs, *places, False)
    return ops._load_hip().moe_combine(y, row, weight, wide)

  def _forward_prefill_sorted(self, flat, weights, selected):
    T, D = flat.shape
    k = self.top_k
    A = T * k
    dev = flat.device
    expert_of = selected.reshape(-1)
    order = torch.argsort(expert_of)
    tok_sorted = torch.arange(T, device=dev).repeat_interleave(k)[order]
    w_sorted = weights.reshape(-1)[order]
    counts = torch.bincount(expert_of, minlength=self.n_experts).cpu().tolist()  # one sync
    xg = flat[tok_sorted]
    ys = []
    off = 0
    for e, c in enumerate(counts):
      if c:
        ys.append(self.experts[e](xg[off:off + c]))
      off += c
    y = torch.cat(ys, dim=0).float() * w_sorted[:, None].float()
    out = torch.zeros(T, D, dtype=torch.float32, device=dev)
    out.index_add_(0, tok_sorted, y)
    return out

  def _forward_decode(self, flat, wide=False):
    """[T, D]; `wide`: fp32, not rounded yet, for a sum with the residual stream."""
    found = self._grouped(flat)
    if found is not None:
      return self._forward_grouped(flat, found, wide)
    T, D = flat.shape
    E, k = self.n_experts, self.top_k
    dev = flat.device
    from xotorch_amd.ops import _load_hip
    hip0 = _load_hip()
    C = max(32, -(-T // 32) * 32)                             # capacity (lossless: count_e <= T)
    if hip0 is not None and flat.is_cuda:
      # fused router (softmax-topk-renorm in one launch)
      logits = self.gate(flat)
      if logits.dtype != torch.bfloat16:
        logits = logits.float()
      selected, weights = hip0.moe_route(logits.contiguous(), None, self.top_k, 0)
    else:
      weights, selected = self._route(flat)                   # [T, k]
    if hip0 is not None and flat.is_cuda:
      # single-launch counting-sort + deterministic combine (replaces the
      # argsort/cumsum/index_add torch glue — measured top MoE decode cost)
      gather_tok, inv_pos = hip0.moe_build(selected.to(torch.int32).contiguous(), E, C)
      scale = None
    else:
      A = T * k
      expert_of = selected.reshape(A)                         # [A]
      token_of = torch.arange(T, device=dev).repeat_interleave(k)
      w_of = weights.reshape(A)
      order = torch.argsort(expert_of)                        # static shape [A]
      sorted_token = token_of[order]
      sorted_w = w_of[order]
      counts = (expert_of.unsqueeze(0) == torch.arange(E, device=dev).unsqueeze(1)).sum(1)
      offsets = torch.cumsum(counts, 0) - counts              # exclusive prefix
      c_idx = torch.arange(C, device=dev)
      pos = offsets.unsqueeze(1) + c_idx.unsqueeze(0)         # [E, C]
      valid = c_idx.unsqueeze(0) < counts.unsqueeze(1)
      pos_c = pos.clamp(max=A - 1)
      gather_tok = sorted_token[pos_c.reshape(-1)]            # [E*C]
      scale = torch.where(valid, sorted_w[pos_c], torch.zeros((), dtype=sorted_w.dtype, device=dev))
    xg = flat.index_select(0, gather_tok)                     # [E*C, D]
    if self.wp_gate_up_fp8 is not None and not torch.is_grad_enabled():
      from xotorch_amd.ops import _load_hip
      hip = _load_hip()
      I = self.intermediate
      x8, sx = hip.quant_fp8_rows(xg)
      gu = hip.skinny_gemm_fp8(x8, sx, self.wp_gate_up_fp8, self.sw_gate_up.view(-1), E, 2 * I)
      h = ops.swiglu_packed(gu.view(E * C, 2 * I))
      h8, sh = hip.quant_fp8_rows(h)
      y = hip.skinny_gemm_fp8(h8, sh, self.wp_down_fp8, self.sw_down.view(-1), E, D)
      y = y.view(E * C, D)
    elif self.wp_gate_up is not None and not torch.is_grad_enabled():
      from xotorch_amd.ops import _load_hip
      hip = _load_hip()
      gu = hip.skinny_gemm_grouped(xg.view(E, C, D), self.wp_gate_up, E, 2 * self.intermediate)
      h = ops.swiglu_packed(gu.view(E * C, 2 * self.intermediate))
      y = hip.skinny_gemm_grouped(h.view(E, C, self.intermediate), self.wp_down, E, D)
      y = y.view(E * C, D)
    else:
      xe = xg.view(E, C, D)
      outs = []
      for e in range(E):
        outs.append(self.experts[e](xe[e]))
      y = torch.cat(outs, dim=0)
    if scale is None:
      return hip0.moe_combine(y.view(E * C, D).to(torch.bfloat16).contiguous(), inv_pos,
                              weights.float().contiguous(), wide)
    out = torch.zeros(T, D, dtype=torch.float32, device=dev)
    out.index_add_(0, gather_tok, y.float() * scale.reshape(-1, 1))
    return out


class DecoderLayer(nn.Module):
  def __init__(self, cfg: ModelConfig):
    super().__init__()
    self.input_layernorm = RMSNorm(cfg.dim, cfg.norm_eps)
    self.self_attn = Attention(cfg)
    self.post_attention_layernorm = RMSNorm(cfg.dim, cfg.norm_eps)
    self.mlp = MoEMLP(cfg) if cfg.n_experts > 0 else MLP(cfg)
    self.eps = cfg.norm_eps

  def _few_rows(self, x) -> bool:
    """Whether all products of this layer are a few rows' (ops.few_rows)."""
    a, m = self.self_attn, self.mlp
    mods = (a.qkv_proj, a.o_proj, m.gate_up_proj, m.down_proj) if type(m) is MLP else ()
    norms = (self.input_layernorm.weight, self.post_attention_layernorm.weight)
    return (len(mods) > 0 and all(type(p) is XotLinear for p in mods)
            and not _watched(a, m, self.input_layernorm, self.post_attention_layernorm, *mods)
            and ops.few_rows_normed(x, norms, *(p.weight for p in mods)))

  def by_tiles(self, x) -> bool:
    """Whether `step` takes this layer: products by weight tiles (ops.tile_rows)."""
    mods = self._modules
    a, before, post = mods["self_attn"], mods["input_layernorm"], mods["post_attention_layernorm"]
    q, o = a._modules["qkv_proj"], a._modules["o_proj"]
    if type(q) is not XotLinear or type(o) is not XotLinear or q.weight_packed_fp8 is not None or o.weight_packed_fp8 is not None:
      return False
    return (x.shape[-1] % 8 == 0 and x.shape[-1] <= 16384 and not _watched(self, a, q, o, post)
            and ops.tiled(x, _own(q), _own(o), wins=ops.parts_win)
            and ops.plain_norms(_own(before), _own(post)))

  def step(self, x, normed, cos, sin, positions, kv, start_pos, is_decode, seq_lens, after):
    """The layer with sums that the next norm finishes: (stream, that norm of it).
    `after`: the module of that norm, or None; normed: this layer's, None: not made yet."""
    mods = self._modules
    a, m, post = mods["self_attn"], mods["mlp"], mods["post_attention_layernorm"]
    if normed is None:
      normed = self.input_layernorm(x)
    qkv, sums = a.project(normed)
    out = a.attend(qkv, cos, sin, positions, kv, start_pos, is_decode, seq_lens, *(() if sums is None else (sums,)))
    follows = after is not None and not _watched(after) and ops.plain_norms(_own(after))
    if type(m) is MLP and m.by_tiles(x) and m.gate_is_tile(x):
      # 45 tokens through 16 layers of 2048: the host took 1171 us a pass for these five calls
      # and their checks, 975 so
      found = ops.tile_rest(out, _own(a._modules["o_proj"]), x, _own(post), post.eps, _own(m._modules["gate_up_proj"]),
                            _own(m._modules["down_proj"]), *((_own(after), after.eps) if follows else ()))
      return found if follows else (found[0], None)
    x, normed = ops.parts_add_norm(ops.tile_parts(out, a.o_proj.weight), x, post.weight, post.eps)
    if type(m) is MLP and m.by_tiles(normed):
      parts = ops.tile_parts(m.gated(normed), m.down_proj.weight)
    elif type(m) is MoEMLP and not _watched(m):
      parts = m._forward_decode(normed.view(-1, x.shape[-1]), True).float()
    else:
      parts = m(normed).float()
    parts = parts.view(-1, x.numel() // x.shape[-1], x.shape[-1])
    if not follows:
      return ops.parts_add_norm(parts, x)[0], None
    return ops.parts_add_norm(parts, x, after.weight, after.eps, rounded=True)

  def forward(self, x, cos, sin, positions, kv, start_pos, is_decode, seq_lens=None):
    if x.shape[0] * x.shape[1] <= ops.FEW_ROWS and kv is not None and self._few_rows(x):
      # norms, activation and residual sums are part of the products
      a, m = self.self_attn, self.mlp
      qkv = ops.rows_norm_linear(x, self.input_layernorm.weight, self.eps, a.qkv_proj.weight, a.qkv_proj.bias)
      out = a.attend(qkv, cos, sin, positions, kv, start_pos, is_decode, seq_lens)
      h = ops.rows_add_linear(out, a.o_proj.weight, x)
      act = ops.rows_norm_swiglu(h, self.post_attention_layernorm.weight, self.eps, m.gate_up_proj.weight)
      return ops.rows_add_linear(act, m.down_proj.weight, h)
    attn_out = self.self_attn(
      self.input_layernorm(x), cos, sin, positions, kv, start_pos, is_decode, seq_lens
    )
    # fused residual-add + norm: h = x + attn_out; normed = rmsnorm(h)
    normed, h = ops.rmsnorm_residual(attn_out, x, self.post_attention_layernorm.weight, self.eps)
    return h + self.mlp(normed)


class ShardedModel(nn.Module):
  """The layer range [shard.start_layer .. shard.end_layer] of one model."""

  def __init__(self, cfg: ModelConfig, shard: Shard):
    super().__init__()
    self.cfg = cfg
    self.shard = shard
    if shard.is_first_layer:
      self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.dim)
    self.layers = nn.ModuleDict({str(i): DecoderLayer(cfg) for i in range(shard.start_layer, shard.end_layer + 1)})
    if shard.is_last_layer:
      self.norm = RMSNorm(cfg.dim, cfg.norm_eps)
      if not cfg.tie_word_embeddings:
        self.lm_head = XotLinear(cfg.dim, cfg.vocab_size, bias=False)
      elif not shard.is_first_layer:
        # tied embeddings but the first shard (owner of embed_tokens) is
        # elsewhere: keep a local copy of the embedding matrix as the head.
        self.lm_head = XotLinear(cfg.dim, cfg.vocab_size, bias=False)
    cos, sin = rope_cos_sin(cfg.head_dim, cfg.max_seq_len, cfg.rope_theta, cfg.rope_scaling)
    self.register_buffer("rope_cos", cos, persistent=False)
    self.register_buffer("rope_sin", sin, persistent=False)

  def reset_rope(self):
    """(Re)compute the fp32 RoPE tables on the current device. Required after
    meta-device construction + to_empty (tables are uninitialized memory)."""
    cos, sin = rope_cos_sin(self.cfg.head_dim, self.cfg.max_seq_len, self.cfg.rope_theta,
                            self.cfg.rope_scaling, device=self.rope_cos.device)
    self.rope_cos = cos
    self.rope_sin = sin

  def _apply(self, fn, recurse=True):
    # keep RoPE tables fp32 (HIP kernel contract): a model-wide .to(bf16)
    # would quantize them; recompute at full precision on the new device.
    super()._apply(fn, recurse)
    if self.rope_cos.device.type != "meta" and self.rope_cos.dtype != torch.float32:
      self.reset_rope()
    return self

  @property
  def local_layer_ids(self) -> List[int]:
    return list(range(self.shard.start_layer, self.shard.end_layer + 1))

  def pack_decode_weights(self, reserve_bytes: int = 8 << 30) -> int:
    """Packs second copies of weights in MFMA fragment order: of what is worth the memory
    (ops.copy_pays; with fp8 weights everything), and of routed experts that grouped products
    do not read as they lie (MoEMLP._expert_weights) - down_proj, lm_head, gate_up, then
    qkv/o - greedily while at least `reserve_bytes` of HBM stay free (KV caches and
    activations are usually allocated before this is called). Returns bytes packed.
    XOT_PACK=none packs nothing, all whatever can be packed and is read."""
    mode = os.getenv("XOT_PACK", "auto")
    if mode == "none" or not torch.cuda.is_available():
      return 0
    groups: List[List[XotLinear]] = [[], [], [], []]
    unread = set()  # experts whose copies nothing would read
    if not ops.fp8_gemm_enabled():
      unread = {id(p) for m in self.modules() if isinstance(m, MoEMLP) and m._expert_weights() is not None
                for e in m.experts for p in (e.gate_up_proj, e.down_proj)}
    for name, mod in self.named_modules():
      if not isinstance(mod, XotLinear) or not mod.packable() or id(mod) in unread:
        continue
      if not ("experts." in name or mode == "all" or ops.fp8_gemm_enabled() or ops.copy_pays(*mod.weight.shape)):
        continue
      if "down_proj" in name:
        # the packed kernel wins when the split-K grid still fills the chip
        # (>= ~1.5 blocks/CU); small-N down projections don't.
        # MoE experts always pack: the grouped launch fills via blockIdx.y.
        if "experts." in name or mod.weight.shape[0] // 128 * 8 >= 384 or mode == "all":
          groups[0].append(mod)
      elif "lm_head" in name:
        groups[1].append(mod)
      elif "gate_up_proj" in name:
        groups[2].append(mod)
      else:  # qkv_proj / o_proj / experts' projections
        groups[3].append(mod)
    if mode != "all" and not ops.fp8_gemm_enabled():
      # default (bf16): qkv/o are not worth the second copy (1.0 of the library's time).
      # In fp8 mode every group wins (half the stream bytes), so all are packed.
      groups = groups[:3]
    packed = 0
    debug = os.getenv("XOT_DEBUG", "0") != "0"
    for gi, grp in enumerate(groups):
      if not grp:
        continue
      bytes_per = 1 if ops.fp8_gemm_enabled() else 2
      need = sum(m.weight.numel() * bytes_per for m in grp)
      free, _ = torch.cuda.mem_get_info()
      if need + reserve_bytes > free:
        if debug:
          print(f"[xot] pack group {gi}: skip (need {need>>20} MiB + reserve "
                f"{reserve_bytes>>20} MiB > free {free>>20} MiB)", flush=True)
        continue
      for m in grp:
        m.pack_decode()
      packed += need
      if debug:
        print(f"[xot] pack group {gi}: packed {len(grp)} modules, {need>>20} MiB", flush=True)
    for mod in self.modules():
      if isinstance(mod, MoEMLP):
        mod.pack_grouped()
    return packed

  def head_weight(self):
    if self.cfg.tie_word_embeddings and hasattr(self, "embed_tokens"):
      return self.embed_tokens.weight
    return self.lm_head.weight

  def forward(
    self,
    x: torch.Tensor,
    caches: List[Tuple[torch.Tensor, torch.Tensor]],
    positions: torch.Tensor,
    start_pos: int,
    is_decode: bool = False,
    seq_lens: Optional[torch.Tensor] = None,
    last_only: bool = True,
  ) -> torch.Tensor:
    """Run this shard.

    x: [B,S] int tokens (first shard) or [B,S,D] hidden states.
    caches: one (k_cache, v_cache) pair per LOCAL layer.
    positions: absolute position ids [S] or [B,S] (device tensor).
    Returns hidden [B,S,D] for non-last shards; logits for the last
    ([B,V] when is_decode/last_only, else [B,S,V]).
    """
    if x.dtype in (torch.int32, torch.int64):
      assert self.shard.is_first_layer, "token input requires the first shard"
      h = self.embed_tokens(x)
    else:
      h = x
    cos, sin = self.rope_cos, self.rope_sin
    # caches=None selects the cache-free training forward; activation
    # checkpointing (on by default when training under grad) trades the
    # per-layer activation residency for a recompute in backward
    use_ckpt = (caches is None and self.training and torch.is_grad_enabled()
                and os.getenv("XOT_ACT_CKPT", "0") == "1")
    layers = [self.layers[str(lid)] for lid in self.local_layer_ids]
    # few enough rows for weight tiles, but not so few that the layers fuse more (ops.few_rows)
    tiles = (caches is not None and h.is_cuda and h.shape[0] * h.shape[1] <= ops.TILE_ROWS and ops.alone(h)
             and not (h.shape[0] * h.shape[1] <= ops.FEW_ROWS and layers[0]._few_rows(h)))
    normed = None
    for idx, layer in enumerate(layers):
      kv = caches[idx] if caches is not None else None
      if tiles and layer.by_tiles(h):
        after = layers[idx + 1].input_layernorm if idx + 1 < len(layers) else None
        if after is None and self.shard.is_last_layer and (h.shape[1] == 1 or not last_only):
          after = self.norm
        h, normed = layer.step(h, normed, cos, sin, positions, kv, start_pos, is_decode, seq_lens, after)
        continue
      normed = None
      if use_ckpt:
        h = torch.utils.checkpoint.checkpoint(
          layer, h, cos, sin, positions, kv, start_pos, is_decode, seq_lens,
          use_reentrant=False)
      else:
        h = layer(h, cos, sin, positions, kv, start_pos, is_decode, seq_lens)
    if not self.shard.is_last_layer:
      return h
    if last_only and h.shape[1] > 1:
      h = h[:, -1:, :].contiguous()  # kernels require contiguous rows
      normed = None
    head = self.head_weight()
    own = self.lm_head if hasattr(self, "lm_head") else None
    if normed is None and (own is None or type(own) is XotLinear) and not (
        _watched(self.norm, *(() if own is None else (own,)))) and (
        ops.few_rows_normed(h, (self.norm.weight,), head)):
      logits = ops.rows_norm_linear(h, self.norm.weight, self.norm.eps, head)
      return logits[:, -1, :] if is_decode or last_only else logits
    h = self.norm(h) if normed is None else normed
    if own is not None:
      logits = own(h)  # XotLinear: packed decode kernel when prepacked
    elif h.numel() <= ops.TILE_ROWS * h.shape[-1] and ops.tile_rows(h, head) and ops.tile_wins(h.numel() // h.shape[-1], *head.shape):
      logits = ops.tile_linear(h, head)
    else:
      logits = ops.linear(h, head.to(h.dtype))
    if is_decode or last_only:
      return logits[:, -1, :]
    return logits


def hf_key_map(shard: Shard, cfg: ModelConfig):
  """Map HF checkpoint keys → this ShardedModel's state-dict keys (shard-aware).

  Packed parameters (fused qkv_proj / gate_up_proj GEMMs) map several HF keys
  to `our_key#part`; the loader concatenates the parts along dim 0 in part
  order. No q/k permute is needed (we use HF's rotate-half RoPE directly).
  """
  mapping = {}
  if shard.is_first_layer:
    mapping["model.embed_tokens.weight"] = "embed_tokens.weight"
  if shard.is_last_layer:
    mapping["model.norm.weight"] = "norm.weight"
    if not cfg.tie_word_embeddings:
      mapping["lm_head.weight"] = "lm_head.weight"
    elif not shard.is_first_layer:
      mapping["model.embed_tokens.weight"] = "lm_head.weight"
  for lid in range(shard.start_layer, shard.end_layer + 1):
    hf = f"model.layers.{lid}."
    ours = f"layers.{lid}."
    for suffix in ("weight",) + (("bias",) if cfg.attn_bias else ()):
      mapping[hf + f"self_attn.q_proj.{suffix}"] = ours + f"self_attn.qkv_proj.{suffix}#0"
      mapping[hf + f"self_attn.k_proj.{suffix}"] = ours + f"self_attn.qkv_proj.{suffix}#1"
      mapping[hf + f"self_attn.v_proj.{suffix}"] = ours + f"self_attn.qkv_proj.{suffix}#2"
    mapping[hf + "self_attn.o_proj.weight"] = ours + "self_attn.o_proj.weight"
    if cfg.qk_norm:
      mapping[hf + "self_attn.q_norm.weight"] = ours + "self_attn.q_norm"
      mapping[hf + "self_attn.k_norm.weight"] = ours + "self_attn.k_norm"
    mapping[hf + "input_layernorm.weight"] = ours + "input_layernorm.weight"
    mapping[hf + "post_attention_layernorm.weight"] = ours + "post_attention_layernorm.weight"
    if cfg.n_experts > 0 and cfg.moe_style == "qwen3":
      mapping[hf + "mlp.gate.weight"] = ours + "mlp.gate.weight"
      for e in range(cfg.n_experts):
        mapping[hf + f"mlp.experts.{e}.gate_proj.weight"] = ours + f"mlp.experts.{e}.gate_up_proj.weight#0"
        mapping[hf + f"mlp.experts.{e}.up_proj.weight"] = ours + f"mlp.experts.{e}.gate_up_proj.weight#1"
        mapping[hf + f"mlp.experts.{e}.down_proj.weight"] = ours + f"mlp.experts.{e}.down_proj.weight"
    elif cfg.n_experts > 0:
      mapping[hf + "block_sparse_moe.gate.weight"] = ours + "mlp.gate.weight"
      for e in range(cfg.n_experts):
        mapping[hf + f"block_sparse_moe.experts.{e}.w1.weight"] = ours + f"mlp.experts.{e}.gate_up_proj.weight#0"
        mapping[hf + f"block_sparse_moe.experts.{e}.w3.weight"] = ours + f"mlp.experts.{e}.gate_up_proj.weight#1"
        mapping[hf + f"block_sparse_moe.experts.{e}.w2.weight"] = ours + f"mlp.experts.{e}.down_proj.weight"
    else:
      mapping[hf + "mlp.gate_proj.weight"] = ours + "mlp.gate_up_proj.weight#0"
      mapping[hf + "mlp.up_proj.weight"] = ours + "mlp.gate_up_proj.weight#1"
      mapping[hf + "mlp.down_proj.weight"] = ours + "mlp.down_proj.weight"
  return mapping
