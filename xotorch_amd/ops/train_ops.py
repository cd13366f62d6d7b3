"""Differentiable forms of the decoder's operators for training on the GPU (bf16,
hip/train_ops.hip, hip/attn_train.hip, hip/gemm_ops.hip): one kernel forward and one backward where separate torch operators
pass fp32 copies through memory. What they cannot take (other types, tracing,
functorch transforms, forward-mode) goes by torch_ref, and so does a backward pass
that is itself differentiated."""
from __future__ import annotations

import os
from typing import Callable, Optional, Sequence

import torch

from xotorch_amd.ops import torch_ref

_ext = _attn = _gemm = _experts = _lora = None
OWN = (torch.Tensor, torch.nn.Parameter)
# looked up once: a step of a small model asks some thirty times
_is_compiling, _is_tracing, _forward_ad = torch.compiler.is_compiling, torch._C._is_tracing, torch.autograd.forward_ad
_dispatch_modes, _transforms = torch._C._len_torch_dispatch_stack, torch._C._are_functorch_transforms_active


def _current_device() -> int:
  return torch._C._cuda_getDevice()


def _hip():
  global _ext
  if _ext is None:
    import importlib
    _ext = importlib.import_module("xotorch_amd.ops._hip_train")
  return _ext


def _hip_attn():
  global _attn
  if _attn is None:
    import importlib
    _attn = importlib.import_module("xotorch_amd.ops._hip_attn_train")
  return _attn


def _hip_gemm():
  global _gemm
  if _gemm is None:
    import importlib
    _gemm = importlib.import_module("xotorch_amd.ops._hip_gemm")
  return _gemm


def _hip_experts():
  global _experts
  if _experts is None:
    import importlib
    _experts = importlib.import_module("xotorch_amd.ops._hip_experts")
  return _experts


def _hip_lora():
  global _lora
  if _lora is None:
    import importlib
    _lora = importlib.import_module("xotorch_amd.ops._hip_lora")
  return _lora


def _missing() -> bool:
  """Whether the kernels are not built and torch's operators are asked for then."""
  if (_ext is None or _attn is None or None in (_gemm, _experts, _lora)) and os.getenv("XOT_ALLOW_EAGER", "0") == "1":
    try:
      _hip(), _hip_attn(), _hip_gemm(), _hip_experts(), _hip_lora()
    except ImportError:
      return True
  return False


def plain(*tensors: torch.Tensor) -> bool:
  """Whether kernels may read these here and now: tensors with memory of their own (fake
  and wrapped ones have none, or another) on the device whose streams launches go to, and
  nobody who follows the operators instead: tracing, a dispatch mode, a functorch
  transform or a forward-mode level, none of which sees a kernel."""
  if not tensors[0].is_cuda or _is_compiling():
    return False
  for t in tensors:
    if type(t) not in OWN:
      return False
  here = _current_device()
  for t in tensors:
    if t.get_device() != here:
      return False
  return not (_dispatch_modes() or _transforms() or _forward_ad._current_level >= 0 or _is_tracing())


def followed() -> bool:
  """Whether somebody follows the operators whom a kernel would lead astray (`plain` without a
  dispatch mode, which sees less then but nothing wrong)."""
  return _is_compiling() or bool(_transforms()) or _forward_ad._current_level >= 0 or bool(_is_tracing())


def takes(x: torch.Tensor, *others: torch.Tensor) -> bool:
  """Whether these operands of a differentiated operator are for the kernels: plain
  bf16 GPU tensors, rows of whole 16 bytes up to 2^17 numbers (norms: up to 16384)."""
  if not (x.is_cuda and torch.is_grad_enabled() and x.dim() > 0 and 0 < x.shape[-1] <= 1 << 17 and x.shape[-1] % 8 == 0 and x.numel() > 0):
    return False
  return (any(t.requires_grad for t in (x, *others)) and all(t.dtype == torch.bfloat16 for t in (x, *others))
          and plain(x, *others) and not _missing())


def once(dy: torch.Tensor, *others: torch.Tensor) -> bool:
  """Whether kernels may take a backward pass with this gradient: nobody differentiates it
  again or follows its operators (which need not be those that followed the forward pass),
  and it is not many gradients at once, which come wrapped and without memory."""
  return not torch.is_grad_enabled() and torch._C._has_storage(dy) and plain(dy, *others)


def _rows(t: torch.Tensor) -> torch.Tensor:
  """Contiguous, with rows on 16 bytes."""
  t = t.contiguous()
  return t if t.data_ptr() % 16 == 0 else t.clone()


def _again(f: Callable, inputs: Sequence[torch.Tensor], needs: Sequence[bool], grads: Sequence) -> list:
  """Gradients of f by torch's own operators, differentiable in turn."""
  with torch.enable_grad():
    outs = f(*inputs)
    outs = outs if isinstance(outs, tuple) else (outs,)
    pairs = [(o, g) for o, g in zip(outs, grads) if g is not None]
    wanted = [t for t, n in zip(inputs, needs) if n]
    found = iter(torch.autograd.grad([o for o, _ in pairs], wanted, [g for _, g in pairs], create_graph=True, allow_unused=True))
  return [next(found) if n else None for n in needs]


# Where the products of hip/gemm_ops.hip are faster than the library's, by what they took of
# its time on the GPU with weights from memory, as a pass finds them (1 to 4096 tokens, the
# linears of decoders of 0.5B to 70B; M tokens through a weight [N, K]). Passes of few tokens or
# short rows wait for the host, to which a call of the library is the longer one: there is no
# lower end, and narrow products of short rows are the kernels' though some are slower by
# themselves. 300 tokens through 28 layers of 1536 took 3070 us, and 3500 with those by the
# library; 512 tokens 3520, and 3420 to 3660. What the kernels don't index is the library's.
_MOST = 1 << 22  # rows, features
_WIDEST = 57344  # of what was measured with tiles of 64 to 224 rows of x


def forward_wins(M: int, N: int, K: int) -> bool:
  """x W^T; the kernels have what this or forward_gains is true for (gradients of inputs: input_wins or
  input_gains). Narrow results of up to 1000 tokens 0.34 to 1.26 (0.77 on average) for rows of 3072
  and more, 0.74 to 1.38 (0.94) for shorter ones (0.76 to 1.65, 1.19, from 65 tokens on before
  there were tiles of 64). By tiles of 128 and 256 alone: wider results and more tokens 0.95 to 1.40, but for long sums, whose library tiles
  fill the chip badly (257 to 2000 tokens by 1536 to 12288 features of 13824 to 29568): where
  the result is small 0.46 to 1.05 (0.69), of up to 6144 features 0.65 to 0.95, narrow ones of
  longest sums 0.39 to 0.87. A vocabulary's width (128256 to 152064 features of 896 to 4096), 65
  to 1000 tokens 0.63 to 1.02 (0.86), from 1333 on 0.92 to 1.05. Above these lines 0.6 to 1.5
  from one size to the next."""
  if K % 64 or N % 4 or max(M, N, K) > _MOST:
    return False
  if N >= 100_000 and K <= 4096:
    return 64 < M <= 1000
  if M <= 1000 and N <= 4096:
    return True
  small = M * N <= 4_300_000 and N <= 12288 or M <= 1000 and N <= 6144
  return M > 256 and (K > 12288 and small or K > 16384 and N <= 4096 and M <= 2000)


def input_wins(M: int, N: int, K: int) -> bool:
  """dy W, a sum over N: 0.22 to 1.11 (0.64 on average), weights of less than 5 10^6 numbers
  0.59 to 1.23 (0.87). By tiles of 128 and 256 alone there was left to the library: by sums of less than four times the
  result's width 1025 to 1400 tokens and weights of 8192 by 8192 and more 1.15 to 1.38, 1281 to
  1400 and smaller ones 0.93 to 1.11 (1.04); 257 to 300 by weights of more than 10^8
  1.21 to 1.43; 3000 by [16384, 2048] 1.15; shorter sums of more tokens 0.85 to 1.27."""
  if N % 64 or K % 8 or max(M, N, K) > _MOST:
    return False
  if M <= 1024:
    return N >= K or M <= (300 if N * K <= 100_000_000 else 256)
  if M <= 1400 and N < 4 * K:
    return N >= K and N * K <= (60_000_000 if M <= 1280 else 8_000_000)
  return M <= 1400 and N >= K or M <= 2800 and N >= 8 * K or M <= 3000 and N >= 10 * K


def forward_gains(M: int, N: int, K: int) -> bool:
  """What is faster of forward_wins' rest since there are tiles of 64 to 224 rows of x: long
  sums 0.27 to 1.15 (0.81; wide ones up to 1000 tokens), narrow ones of the longest, of more
  tokens 0.58 to 1.06 (0.74); small weights 0.68 to 1.07 (0.89); others up to 1000 tokens 0.59 to 1.13 (0.92), up to 2000 0.71 to
  1.12 (0.95). What it leaves: more tokens 0.67 to 1.18 (0.99); 65 to 128 by short sums and by
  wide weights 0.81 to 1.22 (0.98); features and rows that were not measured."""
  if K % 64 or N % 4 or not 896 <= N < 100_000 or not 896 <= K <= _WIDEST or not 64 < M <= 8192:
    return False
  if K > 8000:
    if N <= 6144:
      return M <= 2000 or K > 16384
    if M <= 1000 or K <= 16384:
      return M <= 1000
    # the longest sums, 1001 to 2000 tokens by eight weights of 6400 to 28672 rows: from 10000 rows on 0.59
    # to 1.08 (0.81); fewer rows and up to 1100 tokens 0.57 to 1.13 (0.75), then where blocks of 256 rows by
    # 224 tokens leave up to an eighth of their rounds empty 0.59 to 1.01 (0.80), and 0.53 to 1.16 (0.89)
    # where they leave more
    blocks = -(-N // 256) * -(-M // 224)
    return M <= 1100 or M <= 2000 and (N > 10000 or blocks >= 224 * -(-blocks // 256))
  return 1000 < M if N * K <= 7_000_000 else M <= 2000 and (M > 128 or K > 3200 and N <= 20000)


def input_gains(M: int, N: int, K: int) -> bool:
  """The same of input_wins' rest: up to 2000 tokens 0.47 to 1.11 (0.87), up to 4096 0.48 to 1.09
  (0.88), up to 8192 0.58 to 1.05 (0.90)."""
  return N % 64 == 0 and K % 8 == 0 and 896 <= N < 100_000 and 896 <= K <= _WIDEST and M <= 8192


def weight_wins(M: int, N: int, K: int) -> bool:
  """dy^T x, a sum over tokens: 0.61 to 1.25 (0.88 on average) from 600 tokens on; small weights
  of fewer 0.54 to 1.20 (0.89), large ones and 100 to 512 tokens 0.85 to 1.16."""
  return M >= 64 and N % 8 == 0 and K % 8 == 0 and max(M, N, K) <= _MOST and (M >= 600 or N * K <= 7_000_000)


def product(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
  """x W^T of rows [M, K]"""
  M, (N, K) = x.shape[0], weight.shape
  if (forward_wins(M, N, K) or forward_gains(M, N, K)) and weight.is_contiguous() and weight.data_ptr() % 16 == 0:
    return _hip_gemm().forward(_rows(x), weight)
  return torch.nn.functional.linear(x, weight)


def adapted_product(x: torch.Tensor, weight: torch.Tensor, low: torch.Tensor, by: torch.Tensor, scale: float) -> torch.Tensor:
  """x W^T + scale low by of rows [M, K], fp32 rows [M, rp] and an adapter [rank, N] (hip/lora_ops.hip).
  Added inside the product, the term spares a pass over its result, so that sums of up to 8000 are the
  kernels' up to 8192 tokens: us of 4096 by [28672, 4096], rank 8, the library's product and the pass 732, so
  694; of longer sums the pass is a smaller part: [4096, 14336] 322, 319."""
  M, (N, K) = x.shape[0], weight.shape
  own = forward_wins(M, N, K) or forward_gains(M, N, K) or 2000 < M <= 8192 and forward_gains(2000, N, K) and K <= 8000
  if own and weight.is_contiguous() and weight.data_ptr() % 16 == 0:
    return _hip_gemm().forward(_rows(x), weight, low, by, scale)
  out = torch.nn.functional.linear(x, weight)
  _hip_lora().add(out, low, by, scale)
  return out


def takes_product(x: torch.Tensor, weight: torch.Tensor) -> bool:
  """Whether `product` is a linear of these without a gradient, of more rows than the
  kernels of decode steps take. Prompts by it and gate_product, and by the library, us: 300
  tokens through 16 layers of 2048 1870, 2300; 512 through 28 of 3584 9350, 12430; 1000
  through 16 of 2048 2990, 3370."""
  if not x.is_cuda or x.dtype is not torch.bfloat16 or weight.dtype is not torch.bfloat16 or torch.is_grad_enabled() or weight.dim() != 2:
    return False
  (N, K), M = weight.shape, x.numel() // max(1, weight.shape[1])
  return (256 < M and x.shape[-1] == K and (forward_wins(M, N, K) or forward_gains(M, N, K)) and plain(x, weight)
          and not torch._C._is_any_autocast_enabled() and not _missing())


def gate_wins(M: int, N: int, K: int) -> bool:
  """silu of gate times up in one kernel over the library's product and the activation's
  kernel (0.5B to 70B decoders, 257 to 8192 tokens): 0.64 to 1.00 (0.86 on average), with rows
  of 8192 to 16384 0.75 to 1.10 (0.93) up to 3000 tokens and 1.01 to 1.04 from 4096 on."""
  return M > 256 and K % 64 == 0 and N % 32 == 0 and (K <= 4096 or M <= 3000)


def takes_gate(x: torch.Tensor, weight: torch.Tensor) -> bool:
  """Whether gate_product is for these, without a gradient."""
  if not x.is_cuda or x.dtype is not torch.bfloat16 or weight.dtype is not torch.bfloat16 or torch.is_grad_enabled() or weight.dim() != 2:
    return False
  (N, K), M = weight.shape, x.numel() // max(1, weight.shape[1])
  return (x.shape[-1] == K and max(M, N, K) <= _MOST and gate_wins(M, N, K) and weight.is_contiguous() and weight.data_ptr() % 16 == 0
          and plain(x, weight) and not torch._C._is_any_autocast_enabled() and not _missing())


def gate_product(x: torch.Tensor, gate_up: torch.Tensor) -> torch.Tensor:
  """silu(x gate^T) * (x up^T), products not rounded: gate_up [2 F, K]"""
  return _hip_experts().gate_product(_rows(x.reshape(-1, x.shape[-1])), gate_up).view(*x.shape[:-1], gate_up.shape[0] // 2)


def input_gradient(dy: torch.Tensor, weight: torch.Tensor, low: Optional[torch.Tensor] = None, by: Optional[torch.Tensor] = None) -> torch.Tensor:
  """dy W of rows [M, N], and low by of an adapter [rank, K]"""
  M, (N, K) = dy.shape[0], weight.shape
  if (input_wins(M, N, K) or input_gains(M, N, K)) and once(dy, weight) and weight.is_contiguous() and weight.data_ptr() % 16 == 0:
    return _hip_gemm().input_gradient(_rows(dy), weight, low, by)
  dx = dy @ weight
  if low is not None:
    _hip_lora().add(dx, low, by, 1.0)
  return dx


def weight_gradient(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
  """dy^T x of rows [M, N] and [M, K]"""
  if weight_wins(dy.shape[0], dy.shape[1], x.shape[1]) and once(dy, x):
    return _hip_gemm().weight_gradient(_rows(dy), _rows(x))
  return dy.t() @ x


def takes_linear(x: torch.Tensor, weight: torch.Tensor) -> bool:
  """Whether a linear of these, with a gradient, is one of these products at least."""
  if not (x.is_cuda and torch.is_grad_enabled() and weight.dim() == 2 and 0 < x.numel() and x.shape[-1] == weight.shape[1]):
    return False
  (N, K), M = weight.shape, x.numel() // weight.shape[1]
  return ((forward_wins(M, N, K) or forward_gains(M, N, K) or input_wins(M, N, K) or input_gains(M, N, K) or weight_wins(M, N, K)) and K % 8 == 0
          and x.dtype == weight.dtype == torch.bfloat16 and (x.requires_grad or weight.requires_grad) and plain(x, weight)
          and not torch._C._is_any_autocast_enabled() and not _missing())


class _Linear(torch.autograd.Function):
  """As torch's operator, holds only what its gradients read: a frozen weight's input lives no
  longer than the forward pass."""

  @staticmethod
  def forward(ctx, x, weight):
    need_x, need_weight = ctx.needs_input_grad
    ctx.save_for_backward(x if need_weight else None, weight if need_x else None)
    ctx.shape = x.shape
    return product(x.reshape(-1, x.shape[-1]), weight).view(*x.shape[:-1], weight.shape[0])

  @staticmethod
  def backward(ctx, dy):
    x, weight = ctx.saved_tensors
    rows = dy.reshape(-1, dy.shape[-1])
    dx = input_gradient(rows, weight).view(ctx.shape) if ctx.needs_input_grad[0] else None
    return dx, weight_gradient(rows, x.reshape(-1, x.shape[-1])) if ctx.needs_input_grad[1] else None


def linear(x, weight):
  return _Linear.apply(x, weight)


class _Norm(torch.autograd.Function):
  @staticmethod
  def forward(ctx, x, weight, eps, w_bias):
    from xotorch_amd import ops
    ctx.save_for_backward(x, weight)
    ctx.eps, ctx.w_bias = eps, w_bias
    return ops._load_hip().rmsnorm(_rows(x), _rows(weight), eps, w_bias)

  @staticmethod
  def backward(ctx, dy):
    x, weight = ctx.saved_tensors
    if torch.is_grad_enabled():
      return (*_again(lambda a, b: torch_ref.rmsnorm(a, b, ctx.eps, ctx.w_bias), (x, weight), ctx.needs_input_grad[:2], (dy,)),
              None, None)
    dx, *dw = _hip().norm_backward(_rows(dy), None, _rows(x), None, _rows(weight), ctx.eps, ctx.w_bias, ctx.needs_input_grad[1])
    return dx, dw[0] if dw else None, None, None


class _NormResidual(torch.autograd.Function):
  @staticmethod
  def forward(ctx, x, residual, weight, eps, w_bias):
    from xotorch_amd import ops
    ctx.save_for_backward(x, residual, weight)
    ctx.eps, ctx.w_bias = eps, w_bias
    ctx.set_materialize_grads(False)
    return tuple(ops._load_hip().rmsnorm_residual(_rows(x), _rows(residual), _rows(weight), eps, w_bias))

  @staticmethod
  def backward(ctx, dy, ds):
    x, residual, weight = ctx.saved_tensors
    if dy is None and ds is None:
      return None, None, None, None, None
    if torch.is_grad_enabled():
      return (*_again(lambda a, r, w: torch_ref.rmsnorm_residual(a, r, w, ctx.eps, ctx.w_bias), (x, residual, weight),
                      ctx.needs_input_grad[:3], (dy, ds)), None, None)
    if dy is None:
      return ds, ds, torch.zeros_like(weight) if ctx.needs_input_grad[2] else None, None, None
    dx, *dw = _hip().norm_backward(_rows(dy), None if ds is None else _rows(ds), _rows(x), _rows(residual), _rows(weight),
                                   ctx.eps, ctx.w_bias, ctx.needs_input_grad[2])
    return dx, dx, dw[0] if dw else None, None, None


class _SwiGLU(torch.autograd.Function):
  @staticmethod
  def forward(ctx, gu):
    from xotorch_amd import ops
    ctx.save_for_backward(gu)
    return ops._load_hip().swiglu_packed(_rows(gu))

  @staticmethod
  def backward(ctx, dy):
    gu, = ctx.saved_tensors
    if torch.is_grad_enabled():
      return _again(torch_ref.swiglu_packed, (gu,), (True,), (dy,))[0]
    return _hip().swiglu_backward(_rows(gu), _rows(dy))


def _split(qkv, cos, sin, positions, n_heads, n_kv_heads, hd):
  """The same as _SplitHeads by torch's operators."""
  B, S, _ = qkv.shape
  q, k, v = (t.reshape(B, S, -1, hd) for t in qkv.split([n_heads * hd, n_kv_heads * hd, n_kv_heads * hd], dim=-1))
  q, k = torch_ref.rope_apply(q, k, cos, sin, positions)
  rep = n_heads // n_kv_heads
  return (q.transpose(1, 2).float(), k.transpose(1, 2).repeat_interleave(rep, dim=1).float(),
          v.transpose(1, 2).repeat_interleave(rep, dim=1).float())


class _SplitHeads(torch.autograd.Function):
  @staticmethod
  def forward(ctx, qkv, cos, sin, positions, n_heads, n_kv_heads, hd):
    ctx.save_for_backward(qkv, cos, sin, positions)
    ctx.sizes = n_heads, n_kv_heads, hd
    return tuple(_hip().split_heads(_rows(qkv), cos, sin, positions, n_heads, n_kv_heads, hd))

  @staticmethod
  def backward(ctx, dq, dk, dv):
    qkv, *places = ctx.saved_tensors
    if torch.is_grad_enabled():
      return (_again(lambda t: _split(t, *places, *ctx.sizes), (qkv,), (True,), (dq, dk, dv))[0], *[None] * 6)
    return (_hip().split_heads_backward(_rows(dq), _rows(dk), _rows(dv), *places, ctx.sizes[1]), *[None] * 6)


class _MergeHeads(torch.autograd.Function):
  @staticmethod
  def forward(ctx, out):
    ctx.heads = out.shape[1]
    return _hip().merge_heads(_rows(out))

  @staticmethod
  def backward(ctx, d):
    B, S, width = d.shape
    if torch.is_grad_enabled():
      return d.reshape(B, S, ctx.heads, width // ctx.heads).transpose(1, 2).float()
    return _hip().merge_heads_backward(_rows(d), ctx.heads)


def _attend(qkv, cos, sin, positions, n_heads, n_kv_heads, hd):
  """The same as _CausalHeads by torch's operators, each with a second derivative."""
  q, k, v = _split(qkv, cos, sin, positions, n_heads, n_kv_heads, hd)
  S = q.shape[2]
  scores = (q * hd ** -0.5) @ k.transpose(-1, -2)
  p = scores.masked_fill(torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1), float("-inf")).softmax(-1)
  return (p @ v).to(qkv.dtype).transpose(1, 2).flatten(2)


class _CausalHeads(torch.autograd.Function):
  @staticmethod
  def forward(ctx, qkv, cos, sin, positions, n_heads, n_kv_heads, hd):
    out, *kept = _hip_attn().train_attention(_rows(qkv), cos, sin, positions, n_heads, n_kv_heads, hd)
    ctx.save_for_backward(qkv, cos, sin, positions, *kept)
    ctx.sizes = n_heads, n_kv_heads, hd
    return out

  @staticmethod
  def backward(ctx, dout):
    qkv, cos, sin, positions, *kept = ctx.saved_tensors
    if torch.is_grad_enabled():
      return (_again(lambda t: _attend(t, cos, sin, positions, *ctx.sizes), (qkv,), (True,), (dout,))[0], *[None] * 6)
    return (_hip_attn().train_attention_backward(_rows(dout), _rows(qkv), *kept, cos, sin, positions, *ctx.sizes), *[None] * 6)


def rmsnorm(x, weight, eps: float, w_bias: float = 0.0):
  return _Norm.apply(x, weight, eps, w_bias)


def rmsnorm_residual(x, residual, weight, eps: float, w_bias: float = 0.0):
  return _NormResidual.apply(x, residual, weight, eps, w_bias)


def swiglu_packed(gu):
  return _SwiGLU.apply(gu)


def causal_heads(qkv, cos, sin, positions, n_heads: int, n_kv_heads: int, hd: int):
  """Causal attention of a training pass, fp32 between projection and result:
  [B, S, (H + 2 KVH) hd] -> [B, S, H hd]."""
  if hd in (64, 128) and qkv.shape[0] <= 65535 and qkv.numel() // hd < 1 << 29 and n_heads + 2 * n_kv_heads <= 65535:
    return _CausalHeads.apply(qkv, cos, sin, positions, n_heads, n_kv_heads, hd)
  q, k, v = _SplitHeads.apply(qkv, cos, sin, positions, n_heads, n_kv_heads, hd)
  return _MergeHeads.apply(torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True))


def takes_heads(qkv, cos, sin, positions, hd: int) -> bool:
  """Whether these kernels rotate the heads: tables of a row per token at least, by which
  a sequence longer than them stays torch's to refuse."""
  B, S, _ = qkv.shape
  return (takes(qkv) and hd % 8 == 0 and S <= cos.shape[0] and isinstance(positions, torch.Tensor)
          and positions.dtype == torch.int32 and positions.is_contiguous() and positions.shape in ((S,), (B, S))
          and plain(qkv, cos, sin, positions)
          and all(t.dtype == torch.float32 and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (cos, sin)))
