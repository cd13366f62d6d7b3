"""LoRA adapters for the sharded decoder.

The reference's train CLI is LoRA-flavored (sample data under train/data/lora)
but ships no engine implementation. Here: low-rank A/B
adapters wrap the projection Linears of a ShardedModel; base weights freeze;
merge/unmerge supported for inference; adapter state dicts save/load
separately (small checkpoints).
"""
from __future__ import annotations

import math
from typing import Iterable, List, Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from xotorch_amd.ops import train_ops


def _scaled(a, b, factor: float):
  """factor a @ b, rounded once."""
  return torch.addmm(a.new_empty(()), a, b, beta=0, alpha=factor)


class _Adapted(torch.autograd.Function):
  """x W' + bias + scaling (x A') B' of a frozen W, bf16. The low-rank terms are added by
  their own products onto the full ones, forward and backward: autograd's sum of the two
  ways through and a sum into a tensor of its own each passed all of [.., out] through
  memory once or twice more (4 layers of 4096 with 4096 tokens, rank 16: 15.6 to 15.25 ms)."""

  @staticmethod
  def forward(ctx, x, weight, bias, a, b, scaling):
    rows = x.reshape(-1, x.shape[-1])
    out = F.linear(rows, weight, bias) if bias is not None else train_ops.product(rows, weight)
    low = rows @ a.t()
    out.addmm_(low, b.t(), alpha=scaling)
    ctx.save_for_backward(x, weight, bias, a, b, low)
    ctx.scaling = scaling
    return out.view(*x.shape[:-1], weight.shape[0])

  @staticmethod
  def backward(ctx, dy):
    x, weight, bias, a, b, low = ctx.saved_tensors
    need_x, _, _, need_a, need_b, _ = ctx.needs_input_grad
    if torch.is_grad_enabled():
      dx, da, db = train_ops._again(lambda x, a, b: F.linear(x, weight, bias) + (x @ a.t() @ b.t()) * ctx.scaling, (x, a, b),
                                    (need_x, need_a, need_b), (dy,))
      return dx, None, None, da, db, None
    dy = dy.reshape(-1, dy.shape[-1])
    dlow = _scaled(dy, b, ctx.scaling) if need_x or need_a else None
    dx = train_ops.input_gradient(dy, weight).addmm_(dlow, a).view(x.shape) if need_x else None
    return (dx, None, None, dlow.t() @ x.reshape(-1, x.shape[-1]) if need_a else None,
            _scaled(dy.t(), low, ctx.scaling) if need_b else None, None)


class _AdaptedRows(torch.autograd.Function):
  """The same with fp32 adapters A and B^T by hip/lora_ops.hip: a gradient is read once for both of its
  narrow sums, nothing narrow is rounded but as an operand of their matrix cores; the products of
  hip/gemm_ops.hip add the terms before they store."""

  @staticmethod
  def forward(ctx, x, weight, bias, a, bt, scaling):
    hip, rows = train_ops._hip_lora(), train_ops._rows(x.reshape(-1, x.shape[-1]))
    low, columns = hip.sums(rows, a, 1.0, None, a.shape[0], 1.0, False)
    if bias is None:
      out = train_ops.adapted_product(rows, weight, low, bt, scaling)
    else:
      out = F.linear(rows, weight, bias)
      hip.add(out, low, bt, scaling)
    ctx.save_for_backward(x, weight, bias, a, bt, columns)
    ctx.scaling = scaling
    return out.view(*x.shape[:-1], weight.shape[0])

  @staticmethod
  def backward(ctx, dy):
    x, weight, bias, a, bt, columns = ctx.saved_tensors
    need_x, _, _, need_a, need_b, _ = ctx.needs_input_grad
    if not train_ops.once(dy, x, weight, a, bt):
      def whole(x, a, bt):
        return F.linear(x, weight, bias) + (x @ a.to(x.dtype).t() @ bt.to(x.dtype)) * ctx.scaling
      dx, da, db = train_ops._again(whole, (x, a, bt), (need_x, need_a, need_b), (dy,))
      return dx, None, None, da, db, None
    hip, rank = train_ops._hip_lora(), a.shape[0]
    dy, dx, da, db = train_ops._rows(dy.reshape(-1, dy.shape[-1])), None, None, None
    found = hip.sums(dy, bt if need_x or need_a else None, ctx.scaling, columns if need_b else None, rank, ctx.scaling, False)
    if need_b:
      db = found.pop().t()  # lies as B does
    if need_x:
      dx = train_ops.input_gradient(dy, weight, found[0], a).view(x.shape)
    if need_a:
      da, = hip.sums(train_ops._rows(x.reshape(-1, x.shape[-1])), None, 1.0, found[1], rank, 1.0, True)
    return dx, None, None, da, db, None


class LoRALinear(nn.Module):
  def __init__(self, base: nn.Linear, rank: int = 8, alpha: float = 16.0, dropout: float = 0.0):
    super().__init__()
    self.base = base
    self.rank = rank
    self.scaling = alpha / rank
    # adapters live on the base weight's device, in fp32 (cast per-forward):
    # fp32 master adapters keep LoRA updates stable under bf16 bases
    dev = base.weight.device
    self.lora_a = nn.Parameter(torch.zeros(rank, base.in_features, device=dev, dtype=torch.float32))
    self.lora_b = nn.Parameter(torch.zeros(base.out_features, rank, device=dev, dtype=torch.float32))
    nn.init.kaiming_uniform_(self.lora_a, a=math.sqrt(5))
    self.dropout = nn.Dropout(dropout) if dropout > 0 else nn.Identity()
    self.merged = False
    base.weight.requires_grad_(False)
    if base.bias is not None:
      base.bias.requires_grad_(False)

  def _takes(self, x) -> bool:
    """Whether base and adapter are one function for autograd: plain bf16 GPU tensors, a
    frozen linear of which nobody else sees the result."""
    base = self.base
    if not (x.is_cuda and x.dtype == torch.bfloat16 and torch.is_grad_enabled() and x.numel() > 0
            and type(self.dropout) is nn.Identity and type(base.weight) is nn.Parameter and base.weight.dtype == torch.bfloat16):
      return False
    from xotorch_amd.models.llama import XotLinear
    held = (base.weight,) if base.bias is None else (base.weight, base.bias)
    hooks = (base._forward_hooks, base._forward_pre_hooks, base._backward_hooks, base._backward_pre_hooks,
             self.dropout._forward_hooks, self.dropout._forward_pre_hooks)
    return (type(base) in (nn.Linear, XotLinear) and not any(hooks) and "forward" not in vars(base) and not torch.nn.modules.module._has_any_global_hook()
            and all(t.is_cuda and t.dtype == torch.bfloat16 and not t.requires_grad for t in held)
            and any(t.requires_grad for t in (x, self.lora_a, self.lora_b))
            and not torch.is_autocast_enabled("cuda") and train_ops.plain(x, *held, self.lora_a, self.lora_b))

  def _by_rows(self, x) -> bool:
    """Whether these are for the kernels of narrow sums (_takes holds): for 1 to 300 rows of 4096
    to 28672 numbers both passes took 0.43 to 0.91 of their time by library products (0.64 on
    average), and of the host's, which few rows wait for, 0.48 to 0.85 (0.66)."""
    a, b = self.lora_a, self.lora_b
    return (a.dtype == b.dtype == torch.float32 and a.dim() == b.dim() == 2 and 1 <= a.shape[0] == b.shape[1] <= 16
            and x.shape[-1] == a.shape[1] == self.base.weight.shape[1] and b.shape[0] == self.base.weight.shape[0]
            and a.shape[1] % 256 == 0 and b.shape[0] % 256 == 0
            and max(x.numel() // x.shape[-1], a.shape[1], b.shape[0]) <= train_ops._MOST and not train_ops._missing())

  def forward(self, x):
    if not self.merged and self._takes(x):
      if self._by_rows(x):  # copies: the adapters may change between the passes
        return _AdaptedRows.apply(x, self.base.weight, self.base.bias, self.lora_a.clone(memory_format=torch.contiguous_format),
                                  self.lora_b.t().clone(memory_format=torch.contiguous_format), self.scaling)
      return _Adapted.apply(x, self.base.weight, self.base.bias, self.lora_a.to(x.dtype), self.lora_b.to(x.dtype), self.scaling)
    out = self.base(x)
    if not self.merged:
      if x.is_cuda and x.dtype == out.dtype == torch.bfloat16:
        # the sum and the factor belong to the second product: no pass over [.., out] of their own
        low = (self.dropout(x) @ self.lora_a.to(x.dtype).t()).reshape(-1, self.rank)
        return torch.addmm(out.reshape(-1, out.shape[-1]), low, self.lora_b.to(x.dtype).t(), alpha=self.scaling).view(out.shape)
      lora = self.dropout(x) @ self.lora_a.to(x.dtype).t() @ self.lora_b.to(x.dtype).t()
      out = out + lora * self.scaling
    return out

  @torch.no_grad()
  def merge(self):
    if not self.merged:
      delta = (self.lora_b @ self.lora_a) * self.scaling
      self.base.weight.add_(delta.to(self.base.weight.dtype))
      self.merged = True

  @torch.no_grad()
  def unmerge(self):
    if self.merged:
      delta = (self.lora_b @ self.lora_a) * self.scaling
      self.base.weight.sub_(delta.to(self.base.weight.dtype))
      self.merged = False


DEFAULT_TARGETS = ("qkv_proj", "o_proj", "gate_up_proj", "down_proj")


def apply_lora(model: nn.Module, rank: int = 8, alpha: float = 16.0,
               targets: Iterable[str] = DEFAULT_TARGETS, dropout: float = 0.0) -> List[str]:
  """Wrap matching Linears with LoRALinear; freeze everything else.

  Returns the list of wrapped module paths.
  """
  targets = tuple(targets)
  for p in model.parameters():
    p.requires_grad_(False)
  wrapped = []
  for name, module in list(model.named_modules()):
    for child_name, child in list(module.named_children()):
      if isinstance(child, nn.Linear) and child_name in targets:
        setattr(module, child_name, LoRALinear(child, rank=rank, alpha=alpha, dropout=dropout))
        wrapped.append(f"{name}.{child_name}" if name else child_name)
  return wrapped


def lora_parameters(model: nn.Module):
  return [p for n, p in model.named_parameters() if "lora_" in n]


def lora_state_dict(model: nn.Module) -> dict:
  return {n: p.detach().cpu() for n, p in model.named_parameters() if "lora_" in n}


def load_lora_state_dict(model: nn.Module, sd: dict) -> int:
  own = dict(model.named_parameters())
  n = 0
  with torch.no_grad():
    for name, t in sd.items():
      if name in own:
        own[name].copy_(t.to(own[name].dtype))
        n += 1
  return n
