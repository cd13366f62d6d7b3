"""Prompt attention over the packed cache against 64 bits: rows and keys at the edges of
their tiles (128 rows of heads times positions, 32 and 64 keys), keys split over blocks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pack(k, v):
  """[B, heads, T, 128] -> the fragment order of the cache, T rounded up to 32."""
  B, heads, T, _ = k.shape
  t32 = -(-T // 32) * 32
  k, v = (torch.nn.functional.pad(t, (0, 0, 0, t32 - T)) for t in (k, v))
  return (k.view(B, heads, t32 // 16, 16, 4, 4, 8).permute(0, 1, 2, 4, 5, 3, 6).reshape(B, heads, t32 // 16, 4, 64, 8).contiguous(),
          v.view(B, heads, t32 // 32, 4, 8, 8, 16).permute(0, 1, 5, 2, 3, 6, 4).reshape(B, heads, 8, t32 // 32, 64, 8).contiguous())


@pytest.mark.parametrize("B,S,H,KVH,start,cap,window", [
  (1, 1, 1, 1, 0, 0.0, 0), (2, 33, 5, 1, 31, 0.0, 0), (1, 128, 7, 7, 0, 0.0, 0), (3, 65, 12, 2, 64, 0.0, 0),
  (1, 9, 28, 4, 1500, 0.0, 0), (1, 257, 8, 2, 1023, 0.0, 0), (1, 600, 4, 2, 0, 0.0, 0),
  (1, 140, 4, 2, 300, 20.0, 0), (1, 140, 4, 2, 300, 0.0, 50), (2, 40, 4, 1, 700, 30.0, 64), (1, 300, 2, 1, 0, 0.0, 1)])
def test_prefill_attention(B, S, H, KVH, start, cap, window):
  from xotorch_amd.ops import _hip_ops
  g = torch.Generator(device="cuda").manual_seed(S)
  T, rep = start + S, H // KVH
  qkv = torch.randn(B, S, H + 3, 128, generator=g, device="cuda").to(torch.bfloat16)
  q = qkv[:, :, :H]  # a view of a wider row, as the projection gives it
  k, v = (torch.randn(B, KVH, T, 128, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
  out = _hip_ops.attn_prefill_mfma(q, *_pack(k, v), start, 0.0, cap, window).double()
  kd, vd = k.double().repeat_interleave(rep, 1), v.double().repeat_interleave(rep, 1)
  qd = q.double().transpose(1, 2)
  s = qd @ kd.transpose(-1, -2) * 128 ** -0.5
  # fp32 sums of 128 products, the scaling and the exponent
  off = (qd.abs() @ kd.abs().transpose(-1, -2)).amax(-1, keepdim=True) * 128 ** -0.5 * (132 * 2.0 ** -24)
  if cap:
    s = cap * torch.tanh(s / cap)
  at = torch.arange(start, T, device="cuda")[:, None] - torch.arange(T, device="cuda")[None]
  hidden = (at < 0) | (at >= window) if window else at < 0
  p = s.masked_fill(hidden, -torch.inf).softmax(-1)
  ref, size = (p @ vd).transpose(1, 2), (p @ vd.abs()).transpose(1, 2)
  # probabilities as bf16, above and below the line, and the result
  bound = size * (2.0 ** -7 + 4 * off.transpose(1, 2)) + ref.abs() * 2.0 ** -8
  assert out.shape == ref.shape and bool(((out - ref).abs() <= bound + 1e-6).all())


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("B,S,H,KVH,start", [(1, 5, 4, 1, 2100), (1, 7, 6, 2, 1100), (2, 33, 7, 1, 560), (3, 70, 4, 4, 200), (1, 2000, 12, 2, 0)])
def test_merged_parts(hd, B, S, H, KVH, start):
  """Keys in 2 to 16 parts, one of them past every position that the first tokens see."""
  from xotorch_amd.ops import _hip_ops
  g = torch.Generator(device="cuda").manual_seed(S)
  T, rep = start + S, H // KVH
  t32 = -(-T // 32) * 32
  q, k, v = (torch.randn(*s, hd, generator=g, device="cuda").to(torch.bfloat16) for s in ((B, S, H), (B, KVH, t32), (B, KVH, t32)))
  kp = k.view(B, KVH, t32 // 16, 16, hd // 32, 4, 8).permute(0, 1, 2, 4, 5, 3, 6).reshape(B, KVH, t32 // 16, hd // 32, 64, 8).contiguous()
  vp = v.view(B, KVH, t32 // 32, 4, 8, hd // 16, 16).permute(0, 1, 5, 2, 3, 6, 4).reshape(B, KVH, hd // 16, t32 // 32, 64, 8).contiguous()
  out = _hip_ops.attn_prefill_mfma(q, kp, vp, start, 0.0, 0.0, 0).double()
  kd, vd = (t[:, :, :T].double().repeat_interleave(rep, 1) for t in (k, v))
  s = q.double().transpose(1, 2) @ kd.transpose(-1, -2) * hd ** -0.5
  off = (q.double().abs().transpose(1, 2) @ kd.abs().transpose(-1, -2)).amax(-1, keepdim=True) * hd ** -0.5 * ((hd + 4) * 2.0 ** -24)
  p = s.masked_fill(torch.arange(start, T, device="cuda")[:, None] < torch.arange(T, device="cuda")[None], -torch.inf).softmax(-1)
  ref, size = (p @ vd).transpose(1, 2), (p @ vd.abs()).transpose(1, 2)
  bound = size * (2.0 ** -7 + 4 * off.transpose(1, 2)) + ref.abs() * 2.0 ** -8  # as above
  assert out.shape == ref.shape and bool(((out - ref).abs() <= bound + 1e-6).all())


def test_heads_of_64_in_any_order():
  """Queries whose heads don't lie side by side, or not on 16 bytes."""
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  B, S, H, KVH, start = 2, 40, 4, 2, 7
  g = torch.Generator(device="cuda").manual_seed(0)
  c = ShardKVCache(1, B, KVH, 64, 64, torch.bfloat16, "cuda")[0]
  rows = torch.randn(B, start + S, (H + 2 * KVH) * 64, generator=g, device="cuda").to(torch.bfloat16)
  still, none = torch.ones(start + S, 32, device="cuda"), torch.zeros(start + S, 32, device="cuda")
  ops.rope_qkv_append(rows, still, none, torch.arange(start + S, dtype=torch.int32, device="cuda"), c.k, c.v, H, KVH, 64, c.kp, c.vp)
  q = torch.randn(B, S, H, 64, generator=g, device="cuda").to(torch.bfloat16)
  odd = torch.empty(q.numel() + 4, dtype=torch.bfloat16, device="cuda")[4:].view(q.shape).copy_(q)
  with torch.inference_mode():
    ref = ops.attn_prefill(q, c.k, c.v, start, S, c.kp, c.vp).float()
    for other in (q.transpose(1, 2).contiguous().transpose(1, 2), odd):
      assert not other.is_contiguous() or other.data_ptr() % 16
      out = ops.attn_prefill(other, c.k, c.v, start, S, c.kp, c.vp).float()
      assert bool(((out - ref).abs() <= ref.abs() * 2.0 ** -6 + 2.0 ** -6).all())  # each rounds probabilities and results


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("few,B,S,H,KVH,start,cap,window", [
  # short waves: one step of 32 keys for four of them, 4 and 5 steps, last rows of a block of 32, batches, both options
  (True, 1, 129, 1, 1, 0, 0.0, 0), (True, 1, 19, 7, 1, 108, 0.0, 0), (True, 1, 33, 4, 4, 229, 0.0, 0), (True, 3, 41, 6, 2, 200, 0.0, 0),
  (True, 1, 256, 28, 4, 500, 0.0, 0), (True, 1, 130, 4, 1, 300, 25.0, 0), (True, 2, 140, 4, 2, 300, 0.0, 50), (True, 1, 300, 2, 1, 0, 0.0, 1),
  (True, 1, 70, 4, 1, 600, 30.0, 64),
  # blocks of 128 rows: keys in parts, and whole
  (False, 1, 3, 6, 2, 4000, 0.0, 0), (False, 1, 5, 4, 2, 4000, 0.0, 100), (False, 1, 2, 4, 1, 4100, 20.0, 0),
  (False, 5, 500, 30, 10, 0, 0.0, 0), (False, 11, 140, 40, 8, 70, 0.0, 40), (False, 11, 140, 40, 8, 70, 15.0, 0)])
def test_either_way_of_prompts(hd, few, B, S, H, KVH, start, cap, window):
  from xotorch_amd.ops import _hip_ops
  assert _hip_ops.prefill_few(B, S, H, KVH, hd, start) == few
  g = torch.Generator(device="cuda").manual_seed(S + start)
  T, rep = start + S, H // KVH
  t32 = -(-T // 32) * 32
  q, k, v = (torch.randn(*s, hd, generator=g, device="cuda").to(torch.bfloat16) for s in ((B, S, H), (B, KVH, t32), (B, KVH, t32)))
  kp = k.view(B, KVH, t32 // 16, 16, hd // 32, 4, 8).permute(0, 1, 2, 4, 5, 3, 6).reshape(B, KVH, t32 // 16, hd // 32, 64, 8).contiguous()
  vp = v.view(B, KVH, t32 // 32, 4, 8, hd // 16, 16).permute(0, 1, 5, 2, 3, 6, 4).reshape(B, KVH, hd // 16, t32 // 32, 64, 8).contiguous()
  out = _hip_ops.attn_prefill_mfma(q, kp, vp, start, 0.0, cap, window).double()
  kd, vd = (t[:, :, :T].double().repeat_interleave(rep, 1) for t in (k, v))
  qd = q.double().transpose(1, 2)
  s = qd @ kd.transpose(-1, -2) * hd ** -0.5
  off = (qd.abs() @ kd.abs().transpose(-1, -2)).amax(-1, keepdim=True) * hd ** -0.5 * ((hd + 4) * 2.0 ** -24)
  if cap:
    s = cap * torch.tanh(s / cap)
  at = torch.arange(start, T, device="cuda")[:, None] - torch.arange(T, device="cuda")[None]
  hidden = (at < 0) | (at >= window) if window else at < 0
  p = s.masked_fill(hidden, -torch.inf).softmax(-1)
  ref, size = (p @ vd).transpose(1, 2), (p @ vd.abs()).transpose(1, 2)
  bound = size * (2.0 ** -7 + 4 * off.transpose(1, 2)) + ref.abs() * 2.0 ** -8  # as above
  assert out.shape == ref.shape and bool(((out - ref).abs() <= bound + 1e-6).all())
