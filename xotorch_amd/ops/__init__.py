"""Op dispatch: hand-written CDNA4 HIP kernels on GPU, torch reference on CPU.

The HIP extension (`xotorch_amd.ops.hip`, built in-tree by
`xotorch_amd/ops/build.py` / `__graft_entry__.build()`) owns the per-token
hot path on MI355X. On a GPU box the HIP path is MANDATORY: if a CUDA tensor
reaches an op and the extension is missing, we raise rather than silently
falling back to eager PyTorch (set XOT_ALLOW_EAGER=1 to override for
debugging/ablation only).
"""
from __future__ import annotations

import contextlib
import functools
import os
import threading
from typing import Optional, Tuple

import torch

from xotorch_amd.ops import torch_ref, train_ops

_hip = None
_hip_load_error: Optional[Exception] = None


def _load_hip():
  global _hip, _hip_load_error
  if _hip is not None or _hip_load_error is not None:
    return _hip
  try:
    import importlib
    _hip = importlib.import_module("xotorch_amd.ops._hip_ops")
  except Exception as e:  # extension not built
    _hip_load_error = e
    _hip = None
  return _hip


def hip_available() -> bool:
  return _load_hip() is not None


def _use_hip(*tensors: torch.Tensor) -> bool:
  t = tensors[0]
  if not t.is_cuda:
    return False
  if torch.is_grad_enabled() and any(x.requires_grad for x in tensors):
    # training path: these kernels are inference-only (no autograd); train_ops has
    # differentiable ones for some, the torch ops are differentiable.
    return False
  if _load_hip() is not None:
    return True
  if os.getenv("XOT_ALLOW_EAGER", "0") == "1":
    return False
  raise RuntimeError(
    "xotorch_amd HIP extension is not built but a CUDA tensor reached the op "
    f"dispatch (load error: {_hip_load_error}). Build it with "
    "`python -c \"import __graft_entry__; __graft_entry__.build()\"` or set "
    "XOT_ALLOW_EAGER=1 to explicitly allow the eager fallback."
  )


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float, w_bias: float = 0.0) -> torch.Tensor:
  """w_bias=1.0 gives the gemma convention (scale by 1 + w, fp32 math)."""
  if _use_hip(x, weight) and x.dtype == torch.bfloat16:
    return _hip.rmsnorm(x, weight, eps, w_bias)
  if train_ops.takes(x, weight) and x.shape[-1] <= 16384 and weight.shape == x.shape[-1:]:
    return train_ops.rmsnorm(x, weight, eps, w_bias)
  return torch_ref.rmsnorm(x, weight, eps, w_bias)


def rmsnorm_residual(
  x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float,
  w_bias: float = 0.0
) -> Tuple[torch.Tensor, torch.Tensor]:
  if _use_hip(x, residual, weight) and x.dtype == torch.bfloat16:
    return _hip.rmsnorm_residual(x, residual, weight, eps, w_bias)
  if train_ops.takes(x, residual, weight) and x.shape[-1] <= 16384 and x.shape == residual.shape and weight.shape == x.shape[-1:]:
    return train_ops.rmsnorm_residual(x, residual, weight, eps, w_bias)
  return torch_ref.rmsnorm_residual(x, residual, weight, eps, w_bias)


def rope_apply(q, k, cos, sin, positions):
  """Standalone RoPE (training / oracle paths). On the GPU inference hot
  path RoPE is fused into rope_qkv_append — there is deliberately no
  separate HIP kernel for this op."""
  return torch_ref.rope_apply(q, k, cos, sin, positions)


def rope_qkv_append(qkv, cos, sin, positions, k_cache, v_cache, n_heads: int, n_kv_heads: int,
                    head_dim: int, kp=None, vp=None, q_norm=None, k_norm=None,
                    norm_eps: float = 1e-6, k_scale=None, v_scale=None, sums=None, bias=None):
  """Fused on the packed qkv GEMM output [B,S,(H+2KVH)*hd]: (optionally
  per-head-RMSNorm q/k — qwen3), RoPE-rotate the q heads in place, rotate k
  heads into the cache, copy v heads into the cache. When the MFMA-packed
  cache copies (kp, vp) exist they are appended too. With `sums` (tile_parts) these and
  the bias are the projection, and qkv only receives the queries.
  """
  if _use_hip(qkv) and qkv.dtype == torch.bfloat16:
    _hip.rope_qkv_append(qkv, cos, sin, positions, k_cache, v_cache, n_heads, n_kv_heads, head_dim,
                         kp, vp, q_norm, k_norm, norm_eps, k_scale, v_scale, sums, bias)
    return
  if sums is not None:
    raise ValueError("sums over parts of k are the GPU kernels'")
  torch_ref.rope_qkv_append(qkv, cos, sin, positions, k_cache, v_cache, n_heads, n_kv_heads,
                            head_dim, q_norm, k_norm, norm_eps)


def attn_prefill(q, k_cache, v_cache, start_pos: int, s_len: int, kp=None, vp=None,
                 scale=None, softcap: float = 0.0, window: int = 0):
  if q.is_cuda and q.dtype == torch.bfloat16 and kp is not None and q.shape[3] in (64, 128) \
     and kp.dtype == torch.bfloat16 \
     and (q.shape[3] == 128 or (q.stride(3) == 1 and q.stride(2) == 64 and (q.stride(0) | q.stride(1)) % 8 == 0
                                and q.data_ptr() % 16 == 0)) \
     and os.getenv("XOT_MFMA_ATTN", "1") == "1" and _use_hip(q):
    # causal flash-forward on matrix cores, streaming the MFMA-packed cache (heads of 64
    # in any other order are torch's; of 128 they are refused);
    # softcap/window run gemma2 semantics inside the same kernel (fp8-KV
    # mode keeps prefill on the plain bf16 cache via the sdpa path below)
    return _hip.attn_prefill_mfma(q, kp, vp, start_pos, scale or 0.0, softcap, window)
  if q.is_cuda and not softcap and not window:
    # fallback: sdpa (rocm flash/mem-efficient backends) in model dtype with
    # native GQA — hd != 128 or unpacked-cache path
    import torch.nn.functional as F
    B, S, H, hd = q.shape
    total = start_pos + s_len
    qh = q.transpose(1, 2)
    k = k_cache[:, :, :total]
    v = v_cache[:, :, :total]
    if start_pos == 0:
      out = F.scaled_dot_product_attention(qh, k, v, is_causal=True, enable_gqa=True, scale=scale)
    else:
      mask = torch.ones(S, total, dtype=torch.bool, device=q.device).tril(diagonal=start_pos)
      out = F.scaled_dot_product_attention(qh, k, v, attn_mask=mask, enable_gqa=True, scale=scale)
    return out.transpose(1, 2).contiguous()
  return torch_ref.attn_prefill(q, k_cache, v_cache, start_pos, s_len, scale, softcap, window)


def attn_decode(q, k_cache, v_cache, seq_len, kp=None, vp=None,
                scale=None, softcap: float = 0.0, window: int = 0,
                k_scale=None, v_scale=None):
  """seq_len: int or int32 device tensor [B] (per-sequence lengths).
  With MFMA-packed cache copies (kp, vp) the flash-decoding kernel scores on
  matrix cores (v_mfma_f32_16x16x32_bf16, coalesced 1 KB cache streams).
  softcap/window select gemma2 semantics (MFMA or torch_ref path only)."""
  if _use_hip(q) and q.dtype == torch.bfloat16:
    if not isinstance(seq_len, torch.Tensor):
      seq_len = torch.full((q.shape[0],), int(seq_len), dtype=torch.int32, device=q.device)
    rep = q.shape[2] // k_cache.shape[1]
    if kp is not None and rep <= 16 and q.shape[3] == 128 and os.getenv("XOT_MFMA_ATTN", "1") == "1":
      return _hip.attn_decode_mfma(q, kp, vp, seq_len, k_cache.shape[2],
                                   scale or 0.0, softcap, window, k_scale, v_scale)
    if not softcap and not window and scale is None:
      return _hip.attn_decode(q, k_cache, v_cache, seq_len)
  return torch_ref.attn_decode(q, k_cache, v_cache, seq_len, scale, softcap, window)


_decode_ext = None


def _decode():
  global _decode_ext
  if _decode_ext is None:
    import importlib
    _decode_ext = importlib.import_module("xotorch_amd.ops._hip_decode")
  return _decode_ext


def decode_attends(qkv, n_heads: int, n_kv_heads: int, head_dim: int, kp, *norms) -> bool:
  """Whether decode_attend takes this step: one token a row, a packed bf16 cache of
  head dim 64 or 128, up to 16 heads on a key head. Short rows of many heads of 64 that
  share no keys are done sooner by the separate kernels (16 and 32 heads, 128 to 512 rows
  of up to 128 positions: 13 to 122 us for 13 to 130; 300 and more: 32 to 393 for 34 to 352)."""
  return (qkv.is_cuda and qkv.dtype == torch.bfloat16 and qkv.dim() == 3 and qkv.shape[1] == 1 and qkv.is_contiguous()
          and qkv.data_ptr() % 16 == 0 and kp is not None and kp.dtype == torch.bfloat16 and head_dim in (64, 128)
          and n_heads <= 16 * n_kv_heads and os.getenv("XOT_MFMA_ATTN", "1") == "1"
          and not (head_dim == 64 and n_heads == n_kv_heads and qkv.shape[0] * n_heads >= 2048 and kp.shape[2] <= 8)
          and all(n is None or n.dtype == torch.bfloat16 for n in norms) and _use_hip(qkv))


def decode_attend(qkv, cos, sin, positions, seq_len, k_cache, v_cache, kp, vp, n_heads: int, n_kv_heads: int,
                  q_norm=None, k_norm=None, norm_eps: float = 1e-6, sums=None, bias=None):
  """rope_qkv_append and attn_decode in one: [B, 1, (H+2KVH)*hd] -> [B, 1, H*hd].
  qkv is left as projected; with `sums` (tile_parts) these and the bias are read in its
  place."""
  if not isinstance(seq_len, torch.Tensor):
    seq_len = torch.full((qkv.shape[0],), int(seq_len), dtype=torch.int32, device=qkv.device)
  return _decode().decode_attend(qkv, cos, sin, positions, seq_len, k_cache, v_cache, kp, vp, n_heads, n_kv_heads,
                                 q_norm, k_norm, norm_eps, sums, bias)


def swiglu(gate, up):
  if _use_hip(gate, up) and gate.dtype == torch.bfloat16:
    return _hip.swiglu(gate, up)
  return torch_ref.swiglu(gate, up)


def swiglu_packed(gu):
  """silu(gate)*up on the packed [.., 2I] fused gate_up GEMM output."""
  if _use_hip(gu) and gu.dtype == torch.bfloat16:
    return _hip.swiglu_packed(gu)
  if train_ops.takes(gu) and gu.shape[-1] % 16 == 0:
    return train_ops.swiglu_packed(gu)
  return torch_ref.swiglu_packed(gu)


def geglu_packed(gu):
  """gelu_tanh(gate)*up on the packed [.., 2I] fused gate_up output (gemma2)."""
  if _use_hip(gu) and gu.dtype == torch.bfloat16:
    return _hip.geglu_packed(gu)
  return torch_ref.geglu_packed(gu)


_SKINNY = os.getenv("XOT_SKINNY", "1") == "1"


def pack_decode_weight(w: torch.Tensor) -> torch.Tensor:
  """Pre-shuffle a [N, K] bf16 weight into MFMA A-fragment order for the
  packed skinny decode GEMM: [N/32, K/16, 64 lanes, 8 bf16] with lane =
  (k-half)*32 + n-row. One-time at weight load; coalesced 1 KB wave streams
  at decode."""
  N, K = w.shape
  assert N % 32 == 0 and K % 64 == 0, (N, K)
  return w.view(N // 32, 32, K // 16, 2, 8).permute(0, 2, 3, 1, 4).contiguous()


def pack_decode_weight_fp8(w: torch.Tensor):
  """Quantize a [N, K] weight to OCP e4m3 with per-output-channel scales and
  pre-shuffle into the MFMA fragment order (bytes): returns (packed_uint8,
  s_w fp32 [N]). Half the stream bytes of the bf16 prepack — the W8A8 decode
  GEMM path (XOT_FP8_GEMM=1)."""
  N, K = w.shape
  assert N % 32 == 0 and K % 64 == 0, (N, K)
  s_w = (w.float().abs().amax(dim=1).clamp(min=1e-12) / 448.0)
  w8 = (w.float() / s_w[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
  packed = w8.view(torch.uint8).view(N // 32, 32, K // 16, 2, 8).permute(0, 2, 3, 1, 4).contiguous()
  return packed, s_w.contiguous()


def fp8_gemm_enabled() -> bool:
  return os.getenv("XOT_FP8_GEMM", "0") == "1"


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
  """y = x @ weight^T (+bias) on hipBLASLt/aten.

  The decode hot path uses XotLinear.pack_decode() + skinny_gemm_packed (the
  hand-written CDNA4 weight-streaming MFMA kernel) instead; this is the
  library-GEMM path for prefill/training/CPU and unpacked weights. Training
  passes, and prompts of some hundred tokens, have products of their own where these
  are faster (train_ops.linear, product).
  """
  if bias is None and train_ops.takes_product(x, weight):
    return train_ops.product(x.reshape(-1, x.shape[-1]), weight).view(*x.shape[:-1], weight.shape[0])
  if bias is None and torch.is_grad_enabled() and train_ops.takes_linear(x, weight):
    return train_ops.linear(x, weight)
  return torch.nn.functional.linear(x, weight, bias)


# rows that the kernels of hip/rows_ops.hip take: with 4 (8 layers of llama-3-8b at 8000
# tokens) they took 1018 us and weight tiles 959, with 1 the norm within the product wins
FEW_ROWS = 2
_rows_ext = None


def _rows():
  global _rows_ext
  if _rows_ext is None:
    import importlib
    _rows_ext = importlib.import_module("xotorch_amd.ops._hip_rows")
  return _rows_ext


def alone(*tensors: torch.Tensor) -> bool:
  """Whether a linear of these may be a kernel instead of torch's operator."""
  return train_ops.plain(*tensors) and not torch._C._is_any_autocast_enabled()


class _Sums(threading.local):
  of_more_rows = False


_sums = _Sums()


@contextlib.contextmanager
def sums_of_more_rows():
  """Within this, in this thread, products of one or two rows are summed as those of up to
  16 are (hip/tile_ops.hip, where a row's sums do not depend on the rows beside it), and
  not by the kernels of their own, whose order is another."""
  before, _sums.of_more_rows = _sums.of_more_rows, True
  try:
    yield
  finally:
    _sums.of_more_rows = before


def few_rows(x: torch.Tensor, *weights: torch.Tensor) -> bool:
  """Whether the products of x with these weights ([N, K], bf16) are a few rows'
  (hip/rows_ops.hip): inference on the GPU, up to FEW_ROWS rows, 16-byte rows."""
  if not x.is_cuda or x.dtype != torch.bfloat16 or torch.is_grad_enabled() or not x.is_contiguous() or _sums.of_more_rows:
    return False
  if not 0 < x.numel() <= FEW_ROWS * x.shape[-1] or not alone(x, *weights) or x.data_ptr() % 16 or not _use_hip(x):
    return False
  return all(w.dtype == torch.bfloat16 and w.dim() == 2 and w.shape[1] % 8 == 0 and w.is_contiguous()
             and w.data_ptr() % 16 == 0 and 0 < w.shape[0] <= 1 << 26 for w in weights)


def plain_norms(*norms: torch.Tensor) -> bool:
  """Whether kernels that end or begin with a norm can read these weights."""
  return all(n.is_cuda and n.dtype == torch.bfloat16 and n.is_contiguous() and n.data_ptr() % 16 == 0 for n in norms)


def few_rows_normed(x: torch.Tensor, norms, *weights: torch.Tensor) -> bool:
  """The same where rows like x are normed first, with these weights: they have to fit into LDS."""
  D = x.shape[-1]
  return (few_rows(x, *weights) and (x.numel() // D) * (-(-D // 512) * 1024) <= 128 * 1024
          and plain_norms(*norms))


def rows_linear(x, weight, bias=None):
  return _rows().rows_linear(x, weight, bias)


def rows_norm_linear(x, norm, eps: float, weight, bias=None, w_bias: float = 0.0):
  """rmsnorm(x) @ weight^T + bias"""
  return _rows().rows_norm_linear(x, norm, eps, w_bias, weight, bias)


def rows_norm_swiglu(x, norm, eps: float, gate_up, w_bias: float = 0.0):
  """silu(n @ gate^T) * (n @ up^T) with n = rmsnorm(x), x fp32, products as bf16"""
  return _rows().rows_norm_swiglu(x, norm, eps, w_bias, gate_up)


def rows_add_linear(x, weight, residual):
  """residual + x @ weight^T: an fp32 sum if the residual is bf16, a bf16 one if it
  is fp32 (both addends as bf16)."""
  return _rows().rows_add_linear(x, weight, residual)


# rows that the kernels of hip/tile_ops.hip take
TILE_ROWS = 256
_tile_ext = None


def _tile():
  global _tile_ext
  if _tile_ext is None:
    import importlib
    _tile_ext = importlib.import_module("xotorch_amd.ops._hip_tile")
  return _tile_ext


def tile_rows(x: torch.Tensor, *weights: torch.Tensor) -> bool:
  """Whether the products of x with these weights ([N, K], bf16) go by weight tiles
  (hip/tile_ops.hip): inference on the GPU, up to TILE_ROWS rows, k in steps of 64."""
  return x.is_cuda and alone(x) and tiled(x, *weights)


def tiled(x: torch.Tensor, *weights: torch.Tensor, wins=None) -> bool:
  """The same where the caller has asked whether x is alone; with `wins` (one of the rules
  below) also whether that is the faster way for each of them."""
  if not x.is_cuda or x.dtype is not torch.bfloat16 or torch.is_grad_enabled() or not x.is_contiguous():
    return False
  if not 0 < x.numel() <= TILE_ROWS * x.shape[-1] or x.data_ptr() % 16 or not _use_hip(x):
    return False
  at, rows = x.get_device(), x.numel() // x.shape[-1]
  for w in weights:
    size = w.shape
    if w.dtype is not torch.bfloat16 or len(size) != 2 or size[1] % 64 or not (0 < size[0] <= 1 << 26 and 0 < size[1] <= 1 << 26) \
       or type(w) not in train_ops.OWN or w.get_device() != at or not w.is_contiguous() or w.data_ptr() % 16 \
       or (wins is not None and not wins(rows, size[0], size[1])):
      return False
  return True


@functools.lru_cache(maxsize=1024)
def tile_splits(N: int, K: int) -> int:
  """Parts of k of a product by tiles, as the rules below count them: as few as give some 450
  blocks of 64 weight rows, of 4 steps of 64 at least (splits_of in hip/tile_ops.hip; small
  weights take fewer, parts_of)."""
  return max(1, min(-(-448 // -(-N // 64)), K // 256, 16))


@functools.lru_cache(maxsize=1024)
def gate_splits(N: int, K: int) -> int:
  """The same of the gated product of N weight rows (gate_splits in hip/tile_ops.hip)."""
  tiles = -(-N // 64)
  whole = K <= 1024 or (tiles >= 160 and K <= (2048 if 256 < tiles < 320 else 6144))
  if whole:
    return 1
  n, one, two = tile_splits(N, K), 256 // tiles, 512 // tiles
  if 2 <= one < n and one * tiles >= 200 and N * (K // 64) <= 312500:
    return one
  turned = K <= 16384 and (K % (4096 if n > 1 else 2048) == 0 or (n > 1 and K % n == 0 and K // n % 2048 == 0))
  return two if n < two <= 16 and tiles > 32 and K >= 256 * two and not turned else n


@functools.lru_cache(maxsize=1024)
def _one_round(N: int, K: int) -> bool:
  """Whether k is split in three or more and the blocks of 128 weight rows are no more than
  the chip's 256 CUs. What is split in two has so many rows of x times weight rows that
  fp32 sums take as long as the weights; 288 blocks take as long as 512."""
  splits = tile_splits(N, K)
  return splits >= 3 and -(-N // 128) * splits <= 256


@functools.lru_cache(maxsize=1024)
def _aligned(N: int, K: int) -> bool:
  """Whether rows and parts of k lie a power of two apart, 16 KB or more. Where all blocks begin
  with the same columns they wait for the same few memory channels, and such products took
  1.06 to 1.27 of the library's time up to 64 rows. Since blocks begin at different places
  (first_step in hip/tile_ops.hip) they take 0.48 to 1.03 (0.79 on average), parts 0.28 to 0.98
  (0.69): the line lies where it did before that, on the side of the library."""
  splits = tile_splits(N, K)
  return K >= 8192 and K & (K - 1) == 0 and 1 < splits and splits & (splits - 1) == 0


# The rules below by what was measured over the library's time, for all products of the
# registry's dense decoders with weights from memory (rows 4 to 256).

@functools.lru_cache(maxsize=8192)
def tile_wins(rows: int, N: int, K: int) -> bool:
  """Whether tile_linear is as fast as the library."""
  if rows <= 64 and _aligned(N, K):
    return False
  if rows <= 16:
    return True  # 0.34 to 1.08
  if _one_round(N, K):
    # the sums' own kernel takes 3 us and more. Up to 64 rows 0.25 to 1.05; up to 128 0.27
    # to 1.11, smaller weights to 1.59; up to 256 0.36 to 1.11, smaller ones to 1.68
    return rows <= 64 or N * K >= (9_000_000 if rows <= 128 else 16_500_000)
  # not split: 0.67 to 1.14 (0.95 on average) up to 64 rows, 0.75 to 1.19 (1.01) up to 128,
  # 1.26 on average above; split, but in more than a round 1.07, 1.11 and 1.26 on average
  return rows <= 64 and tile_splits(N, K) == 1


@functools.lru_cache(maxsize=8192)
def parts_win(rows: int, N: int, K: int) -> bool:
  """The same for tile_parts, whose sums the next kernel adds up: 0.23 to 1.21 (0.7 on
  average) up to 16 rows, then 0.23 to 1.08 in one round; in more 0.72 to 1.15 up to 64
  rows, 0.72 to 1.54 above, by which layers of mistral-large and
  llama-3.1-405b took 1.03 to 1.14 of what they take by the library."""
  return rows <= 16 or _one_round(N, K) or (rows <= 64 and not _aligned(N, K))


@functools.lru_cache(maxsize=8192)
def gate_wins(rows: int, N: int, K: int) -> bool:
  """The same for tile_swiglu, beside the library and the activation's kernel: 0.36 to 1.21
  (0.88 on average) up to 64 rows, 0.75 to 1.16 (0.97) up to 128 but split in two and in
  more than a round 0.78 to 1.28 (1.09). With 136 rows and more 0.77 to 1.01 (0.88) where
  a weight tile makes one round of the chip (gate_tile in hip/tile_ops.hip), 0.66 to 0.96
  (0.81) where rows are short and whole, but 1.03 to 1.25 of 17920, which just pass a round of
  64 each; else 0.97 to 1.57; from 256 weight rows a tile gains nothing on the
  library at 129."""
  if rows <= 64:
    return True
  whole = gate_splits(N, K) == 1 and not 16384 < N < 20480
  if rows <= 128:
    return whole or tile_splits(N, K) != 2 or -(-N // 128) * 2 <= 256
  if whole and K <= 2048 and 6144 <= N <= 24576:
    return True
  return rows >= 136 and tile_splits(N, K) == 1 and any(199 * t < N <= 256 * t for t in (128, 160, 256))


def copy_pays(N: int, K: int) -> bool:
  """Whether a copy of bf16 weights in fragment order (pack_decode_weight) is worth its
  memory: products that tiles do in one round never read it, and below 2.5 10^8 numbers it
  took 0.77 to 1.31 of the library's time with 32 and 64 rows, which the gated tile or the
  plain one came close to or passed (24576 to 37888 rows of 3584 to 5120: 0.9 to 1.03 beside
  0.83 to 1.09, with the activation inside). Above, 0.65 to 1.07 with 32 to 128 rows."""
  return N * K >= 250_000_000 and not _one_round(N, K)


def tile_parted(weight, bias=None) -> bool:
  """Whether tile_linear would split k and add its parts up in a kernel of its own."""
  N, K = weight.shape
  return N % 4 == 0 and (bias is None or bias.dtype == torch.bfloat16) and tile_splits(N, K) > 1


def tile_linear(x, weight, bias=None):
  return _tile().tile_linear(x, weight, bias)


def tile_swiglu(x, gate_up):
  """silu(x @ gate^T) * (x @ up^T), products as bf16"""
  return _tile().tile_swiglu(x, gate_up)


def tile_parts(x, weight):
  """x @ weight^T as fp32 sums over parts of k [parts, rows, N]"""
  return _tile().tile_parts(x, weight)


def parts_add_norm(parts, x, norm=None, eps: float = 0.0, w_bias: float = 0.0, rounded: bool = False):
  """(h, rmsnorm(h)) with h = x + the parts' sum as bf16; (h,) without a norm.
  rounded: the norm reads h as bf16."""
  return _tile().parts_add_norm(parts, x, norm, eps, w_bias, rounded)


def tile_rest(heads, wo, x, post, post_eps: float, gate_up, down, after=None, after_eps: float = 0.0):
  """parts_add_norm, tile_swiglu and parts_add_norm again behind a layer's attention, one
  call from Python: (h, rmsnorm(h) as the next layer wants it), (h,) without a next norm."""
  return _tile().tile_rest(heads, wo, x, post, post_eps, gate_up, down, after, after_eps)


def load_library(device, dtype: torch.dtype):
  """Has the GEMM library load its kernels of this type, which takes 0.35 s once (1.1 with
  bench.py's table of tuned products). Decode steps don't use it: without this the first
  prompt would wait."""
  a = torch.zeros(512, 512, device=device, dtype=dtype)
  torch.nn.functional.linear(a, a)


def softmax_sample(logits, temperature: float = 0.0, top_k: int = 0, generator=None,
                   top_p: float = 0.0):
  # torch ops here are graph-capturable (argmax / exponential+argmax)
  return torch_ref.softmax_sample(logits, temperature, top_k, generator, top_p)
