"""A decode step's attention from the projection on (hip/decode_attn.hip): against 64 bits,
and its caches against the separate append. Lengths at the edges of tiles (32), rows long
enough for several blocks, parked rows, rows that share a position."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [  # B, H, KVH, hd, T, lengths (the new position included), norms, shared position
  (1, 1, 1, 64, 8, [1], False, True), (2, 8, 2, 64, 100, [32, 33], False, False), (1, 32, 8, 64, 1024, [221], False, True),
  (3, 16, 1, 128, 70, [64, 65, 1], True, False), (2, 28, 4, 128, 4096, [3100, 7], False, False),
  (4, 5, 1, 64, 2400, [2400, 1, 1500, 800], True, False), (70, 8, 8, 128, 96, [40] * 70, False, True),
  (2, 12, 2, 128, 2050, [2050, 257], True, False)]


@pytest.mark.parametrize("B,H,KVH,hd,T,lens,norms,shared", CASES)
def test_decode_attend(B, H, KVH, hd, T, lens, norms, shared):
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  from xotorch_amd.ops import torch_ref
  g = torch.Generator(device="cuda").manual_seed(T)

  def rand(*shape):
    return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)

  cos, sin = torch_ref.rope_cos_sin(hd, T, 10000.0, device="cuda")
  caches = [ShardKVCache(1, B, KVH, T, hd, torch.bfloat16, "cuda")[0] for _ in range(2)]
  old = rand(B, T, (H + 2 * KVH) * hd)
  at = torch.arange(T, dtype=torch.int32, device="cuda")
  for c in caches:
    ops.rope_qkv_append(old.clone(), cos, sin, at, c.k, c.v, H, KVH, hd, c.kp, c.vp)
  qkv = rand(B, 1, (H + 2 * KVH) * hd)
  qn, kn = (rand(hd), rand(hd)) if norms else (None, None)
  seen = torch.tensor(lens, dtype=torch.int32, device="cuda")
  pos = (seen[:1] if shared else seen) - 1
  assert ops.decode_attends(qkv, H, KVH, hd, caches[0].kp, qn, kn)
  before = qkv.clone()
  out = ops.decode_attend(qkv, cos, sin, pos, seen, *caches[0][:4], H, KVH, qn, kn, 1e-6)
  assert torch.equal(qkv, before)
  ops.rope_qkv_append(qkv, cos, sin, pos, caches[1].k, caches[1].v, H, KVH, hd, caches[1].kp, caches[1].vp, qn, kn, 1e-6)
  # fp32 sums of the norm in another order: a step of bf16 at most, and that rarely
  for a, b in zip(caches[0][:4], caches[1][:4]):
    assert torch.equal(a, b) if not norms else bool(((a.float() - b.float()).abs() <= b.float().abs() * 2.0 ** -7).all())
  q = qkv[:, 0, :H * hd].view(B, H, hd).double()
  for b, n in enumerate(lens):
    k, v = (c[b, :, :n].double().repeat_interleave(H // KVH, 0) for c in (caches[0].k, caches[0].v))
    s = (k @ q[b, :, :, None])[..., 0] * hd ** -0.5
    # fp32 sums of hd products; with norms a query may be a step of bf16 off as well
    off = (k.abs() @ q[b, :, :, None].abs())[..., 0].amax(-1, keepdim=True) * hd ** -0.5 * ((hd + 4) * 2.0 ** -24 + (2.0 ** -8 if norms else 0))
    p = s.softmax(-1)
    ref, size = (p[:, None] @ v)[:, 0], (p[:, None] @ v.abs())[:, 0]
    bound = size * (2.0 ** -7 + 4 * off) + ref.abs() * 2.0 ** -8
    assert bool(((out[b, 0].view(H, hd).double() - ref).abs() <= bound + 1e-6).all())


@pytest.mark.parametrize("B,S,H,KVH,hd,n,bias,norms", [(1, 1, 1, 1, 64, 1, False, False), (3, 1, 28, 4, 128, 7, True, False),
                                                       (2, 1, 16, 1, 64, 16, True, True), (5, 1, 8, 8, 128, 5, False, True),
                                                       (1, 45, 32, 8, 64, 9, False, False), (2, 33, 7, 1, 128, 4, True, True),
                                                       (3, 71, 32, 8, 128, 3, True, False), (2, 99, 32, 8, 64, 2, False, False),
                                                       (130, 1, 4, 4, 128, 2, True, False)])
def test_sums_over_parts_of_k(B, S, H, KVH, hd, n, bias, norms):
  """The same numbers as from the tensor that they add up to, in order, rounded."""
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  from xotorch_amd.ops import torch_ref
  g = torch.Generator(device="cuda").manual_seed(n)
  T, width = 300, (H + 2 * KVH) * hd
  cos, sin = torch_ref.rope_cos_sin(hd, T, 10000.0, device="cuda")
  sums = torch.randn(n, B * S, width, generator=g, device="cuda")
  b = torch.randn(width, generator=g, device="cuda").to(torch.bfloat16) if bias else None
  qn, kn = (torch.randn(hd, generator=g, device="cuda").to(torch.bfloat16) for _ in "qk") if norms else (None, None)
  total = sums[0].clone()
  for s in sums[1:]:
    total += s
  qkv = (total + b.float() if bias else total).to(torch.bfloat16).view(B, S, width)
  pos = torch.arange(200, 200 + S, dtype=torch.int32, device="cuda")
  found = []
  for parts in (False, True):
    c = ShardKVCache(1, B, KVH, T, hd, torch.bfloat16, "cuda")[0]
    given, more = (torch.full_like(qkv, float("nan")), (sums, b)) if parts else (qkv.clone(), ())
    if S == 1:
      seen = torch.full((B,), 201, dtype=torch.int32, device="cuda")
      out = ops.decode_attend(given, cos, sin, pos, seen, *c[:4], H, KVH, qn, kn, 1e-6, *more)
    else:
      ops.rope_qkv_append(given, cos, sin, pos, c.k, c.v, H, KVH, hd, c.kp, c.vp, qn, kn, 1e-6, None, None, *more)
      out = given[..., :H * hd]
    found.append((out, *c[:4]))
  for x, y in zip(*found):
    assert torch.equal(x, y)


@pytest.mark.parametrize("start", [0, 8, 13])
@pytest.mark.parametrize("B,S,H,KVH,hd,spread", [(1, 1027, 6, 3, 128, False), (3, 700, 7, 2, 64, False), (2, 515, 9, 3, 128, True), (20, 61, 5, 2, 128, False),
                                                 (2, 1024, 5, 2, 64, True)])
def test_values_turned_among_lanes(B, S, H, KVH, hd, spread, start):
  """Eight channels a lane, values of eight positions written at once where they lie side by side, against a
  wave a token: starts on and off a multiple of eight, sequences that end within one, shorter ones than a run has."""
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  T = S + 70
  g = torch.Generator(device="cuda").manual_seed(S + start)
  ones, zeros = torch.ones(T, hd // 2, device="cuda"), torch.zeros(T, hd // 2, device="cuda")
  qkv = torch.randn(B, S, (H + 2 * KVH) * hd, generator=g, device="cuda").to(torch.bfloat16)
  pos = torch.arange(start, start + S, dtype=torch.int32, device="cuda")
  if spread:
    pos = torch.stack([pos + 8 * b + (b > 0) for b in range(B)])
  found = []
  for step in (S, 4):
    c = ShardKVCache(1, B, KVH, T, hd, torch.bfloat16, "cuda")[0]
    queries = []
    for at in range(0, S, step):
      part = qkv[:, at:at + step].clone()
      ops.rope_qkv_append(part, ones, zeros, pos[..., at:at + step].contiguous(), c.k, c.v, H, KVH, hd, c.kp, c.vp)
      queries.append(part[..., :H * hd])
    found.append((torch.cat(queries, 1), *c[:4]))
  assert all(torch.equal(x, y) for x, y in zip(*found))


@pytest.mark.parametrize("what", ["kp as rows", "vp of fewer positions", "kp of fewer sequences", "copies of fewer positions", "caches of fewer heads",
                                  "values of fewer positions", "scales of fewer positions", "fp32 caches"])
def test_caches_that_kernels_would_write_past(what):
  """Refused on the host, before anything is launched: sizes that the kernels' indexes do not fit."""
  from xotorch_amd.ops import _hip_ops
  B, S, H, KVH, hd, T = 2, 40, 4, 2, 128, 64
  f8 = what.startswith("scales")
  make = lambda *size, dtype=torch.bfloat16: torch.zeros(*size, dtype=dtype, device="cuda")
  kc, vc = make(B, KVH, T, hd), make(B, KVH, T, hd)
  kp, vp = (make(*size, 64, 8, dtype=torch.uint8 if f8 else torch.bfloat16) for size in ((B, KVH, T // 16, hd // 32), (B, KVH, hd // 16, T // 32)))
  scales = [make(B, KVH, T, dtype=torch.float32) for _ in range(2)] if f8 else [None, None]
  if what == "kp as rows":
    kp = make(B, KVH, T, hd)
  elif what == "vp of fewer positions":
    vp = vp[:, :, :, :1].contiguous()
  elif what == "kp of fewer sequences":
    kp = kp[:1]
  elif what == "copies of fewer positions":
    kp, vp = kp[:, :, :2].contiguous(), vp[:, :, :, :1].contiguous()
  elif what == "caches of fewer heads":
    kc, vc = kc[:, :1].contiguous(), vc[:, :1].contiguous()
  elif what == "values of fewer positions":
    vc = vc[:, :, :48].contiguous()
  elif what == "fp32 caches":
    kc, vc = kc.float(), vc.float()
  else:
    scales[1] = scales[1][:, :, :32].contiguous()
  qkv, at = make(B, S, (H + 2 * KVH) * hd), torch.arange(S, dtype=torch.int32, device="cuda")
  table = make(T, hd // 2, dtype=torch.float32)
  with pytest.raises(RuntimeError):
    _hip_ops.rope_qkv_append(qkv, table, table, at, kc, vc, H, KVH, hd, kp, vp, k_scale=scales[0], v_scale=scales[1])
  if what not in ("copies of fewer positions", "caches of fewer heads", "values of fewer positions", "fp32 caches"):
    with pytest.raises(RuntimeError):
      _hip_ops.attn_decode_mfma(make(B, 1, H, hd), kp, vp, torch.full((B,), 20, dtype=torch.int32, device="cuda"), T, k_scale=scales[0], v_scale=scales[1])


@pytest.mark.parametrize("B,S,H,KVH,hd,per_row,norms", [(1, 1027, 4, 1, 128, False, True), (3, 333, 30, 2, 64, True, False),
                                                        (2, 515, 9, 3, 128, True, True)])
def test_rows_of_prompts_as_one_by_one(B, S, H, KVH, hd, per_row, norms):
  """Many tokens, several to a wave, against a wave a token (few of them at a time)."""
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  from xotorch_amd.ops import torch_ref
  g = torch.Generator(device="cuda").manual_seed(S)
  T = S + 70
  cos, sin = torch_ref.rope_cos_sin(hd, T, 10000.0, device="cuda")
  qkv = torch.randn(B, S, (H + 2 * KVH) * hd, generator=g, device="cuda").to(torch.bfloat16)
  qn, kn = (torch.randn(hd, generator=g, device="cuda").to(torch.bfloat16) for _ in "qk") if norms else (None, None)
  pos = torch.arange(5, 5 + S, dtype=torch.int32, device="cuda")
  if per_row:
    pos = torch.stack([pos + 17 * b for b in range(B)])
  found = []
  for step in (S, 16):
    c = ShardKVCache(1, B, KVH, T, hd, torch.bfloat16, "cuda")[0]
    queries = []
    for at in range(0, S, step):
      part = qkv[:, at:at + step].clone()
      ops.rope_qkv_append(part, cos, sin, pos[..., at:at + step].contiguous(), c.k, c.v, H, KVH, hd, c.kp, c.vp, qn, kn, 1e-6)
      queries.append(part[..., :H * hd])
    found.append((torch.cat(queries, 1), *c[:4]))
  for n, (x, y) in enumerate(zip(*found)):
    # values as they are; x cos - y sin may be contracted either way, which is off by 2^-23 of
    # terms up to 8 and a step of bf16 then, rarely; a norm's sums are in another order
    if n in (2, 4):
      assert torch.equal(x, y)
    assert bool(((x.float() - y.float()).abs() <= y.float().abs() * 2.0 ** -7 + 2.0 ** -20).all())
    assert (x != y).float().mean() < 0.01


def test_parked_row_keeps_to_its_own_place():
  """A row that sees less than its position appends there and reads what it sees."""
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  from xotorch_amd.ops import torch_ref
  cos, sin = torch_ref.rope_cos_sin(128, 256, 10000.0, device="cuda")
  c = ShardKVCache(1, 2, 2, 256, 128, torch.bfloat16, "cuda")[0]
  g = torch.Generator(device="cuda").manual_seed(0)
  qkv = torch.randn(2, 1, 8 * 128, generator=g, device="cuda").to(torch.bfloat16)
  c.v[:, :, 0] = 1.0
  c.vp.view(2, 2, 8, 8, 64, 8)[:, :, :, 0, :16, 0] = 1.0
  pos, seen = torch.tensor([255, 300], dtype=torch.int32, device="cuda"), torch.tensor([1, 0], dtype=torch.int32, device="cuda")
  cos, sin = (torch.cat([t, t]) for t in (cos, sin))
  out = ops.decode_attend(qkv, cos, sin, pos, seen, *c[:4], 4, 2)
  assert torch.equal(out[0], torch.ones_like(out[0])) and torch.equal(out[1], torch.zeros_like(out[1]))
  assert torch.equal(c.v[0, :, 255].flatten(), qkv[0, 0, 6 * 128:]) and not c.v[0, :, 1:255].any() and not c.v[1, :, 1:].any()


@pytest.mark.parametrize("S,H,KVH,start", [(1, 4, 2, 0), (45, 32, 8, 0), (257, 8, 2, 1000), (130, 7, 1, 63)])
def test_prompt_attention_of_64_channels(S, H, KVH, start):
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  g = torch.Generator(device="cuda").manual_seed(S)
  c = ShardKVCache(1, 2, KVH, start + S, 64, torch.bfloat16, "cuda")[0]
  qkv = torch.randn(2, start + S, (H + 2 * KVH) * 64, generator=g, device="cuda").to(torch.bfloat16)
  still, none = torch.ones(start + S, 32, device="cuda"), torch.zeros(start + S, 32, device="cuda")
  ops.rope_qkv_append(qkv, still, none, torch.arange(start + S, dtype=torch.int32, device="cuda"), c.k, c.v, H, KVH, 64, c.kp, c.vp)
  q = qkv[:, start:, :H * 64].reshape(2, S, H, 64)
  with torch.no_grad():
    out = ops.attn_prefill(q, c.k, c.v, start, S, c.kp, c.vp).double()
  k, v = (t.double().repeat_interleave(H // KVH, 1) for t in (c.k, c.v))
  s = q.double().transpose(1, 2) @ k.transpose(-1, -2) * 64 ** -0.5
  later = torch.arange(start + S, device="cuda")[None] > torch.arange(start, start + S, device="cuda")[:, None]
  p = s.masked_fill(later, -torch.inf).softmax(-1)
  ref, size = (p @ v).transpose(1, 2), (p @ v.abs()).transpose(1, 2)
  assert bool(((out - ref).abs() <= size * 2.0 ** -7 * 1.05 + ref.abs() * 2.0 ** -8 + 1e-6).all())


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("place", [300, -3])
def test_parked_row_reads_within_the_tables(hd, place):
  """Tables of as many rows as the cache has positions: a row that stands elsewhere is
  not appended, and turned by the nearest row that they have."""
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  from xotorch_amd.ops import torch_ref
  T, H, KVH, n = 256, 4, 2, 64
  g = torch.Generator(device="cuda").manual_seed(1)
  cos, sin = torch_ref.rope_cos_sin(hd, T, 10000.0, device="cuda")
  c = ShardKVCache(1, 1, KVH, T, hd, torch.bfloat16, "cuda")[0]
  rows = torch.randn(1, n, (H + 2 * KVH) * hd, generator=g, device="cuda").to(torch.bfloat16)
  ops.rope_qkv_append(rows, cos, sin, torch.arange(n, dtype=torch.int32, device="cuda"), c.k, c.v, H, KVH, hd, c.kp, c.vp)
  qkv = torch.randn(1, 1, (H + 2 * KVH) * hd, generator=g, device="cuda").to(torch.bfloat16)
  before = [t.clone() for t in c[:4]]
  out = ops.decode_attend(qkv, cos, sin, torch.tensor([place], dtype=torch.int32, device="cuda"),
                          torch.tensor([n], dtype=torch.int32, device="cuda"), *c[:4], H, KVH)
  assert all(torch.equal(a, b) for a, b in zip(c[:4], before))
  at = min(max(place, 0), T - 1)
  q = qkv[0, 0, :H * hd].view(H, hd).double()
  q1, q2 = q.chunk(2, -1)
  q = torch.cat([q1 * cos[at] - q2 * sin[at], q2 * cos[at] + q1 * sin[at]], -1)
  k, v = (t[0, :, :n].double().repeat_interleave(H // KVH, 0) for t in (c.k, c.v))
  s = (k @ q[..., None])[..., 0] * hd ** -0.5
  off = (k.abs() @ q.abs()[..., None])[..., 0].amax(-1, keepdim=True) * hd ** -0.5 * 2.0 ** -8  # queries are rounded
  p = s.softmax(-1)
  ref, size = (p[:, None] @ v)[:, 0], (p[:, None] @ v.abs())[:, 0]
  assert bool(((out.view(H, hd).double() - ref).abs() <= size * (2.0 ** -7 + 4 * off) + ref.abs() * 2.0 ** -8).all())


@pytest.mark.parametrize("hd,T", [(64, 64), (64, 3000), (128, 3000)])
def test_nan_is_seen(hd, T):
  """A query that is not a number gives outputs that are not, in one block or several."""
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  H, KVH = 4, 1
  c = ShardKVCache(1, 1, KVH, T, hd, torch.bfloat16, "cuda")[0]
  still, none = torch.ones(T, hd // 2, device="cuda"), torch.zeros(T, hd // 2, device="cuda")
  qkv = torch.ones(1, 1, (H + 2 * KVH) * hd, device="cuda", dtype=torch.bfloat16)
  qkv[0, 0, hd] = float("nan")
  at = torch.tensor([T - 1], dtype=torch.int32, device="cuda")
  out = ops.decode_attend(qkv, still, none, at, at + 1, *c[:4], H, KVH).view(H, hd)
  assert bool(out[1].isnan().all()) and bool(torch.isfinite(out[[0, 2, 3]]).all())


@pytest.mark.parametrize("B,H,KVH,T,n", [(1, 32, 8, 256, 221), (3, 16, 1, 96, 65), (1, 8, 2, 7000, 6999)])
def test_probabilities_of_64_channels_stay_fp32(B, H, KVH, T, n):
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  g = torch.Generator(device="cuda").manual_seed(n)
  c = ShardKVCache(1, B, KVH, T, 64, torch.bfloat16, "cuda")[0]
  still, none = torch.ones(T, 32, device="cuda"), torch.zeros(T, 32, device="cuda")
  rows = torch.randn(B, n, (H + 2 * KVH) * 64, generator=g, device="cuda").to(torch.bfloat16)
  ops.rope_qkv_append(rows.clone(), still, none, torch.arange(n, dtype=torch.int32, device="cuda"), c.k, c.v, H, KVH, 64, c.kp, c.vp)
  qkv = rows[:, -1:].contiguous()
  at = torch.full((B,), n - 1, dtype=torch.int32, device="cuda")
  out = ops.decode_attend(qkv, still, none, at, at + 1, *c[:4], H, KVH).view(B, KVH, H // KVH, 64).double()
  q = qkv[:, 0, :H * 64].view(B, KVH, H // KVH, 64).double()
  k, v = c.k[:, :, :n].double(), c.v[:, :, :n].double()
  s = q @ k.transpose(-1, -2).contiguous() * 0.125
  off = (q.abs() @ k.abs().transpose(-1, -2).contiguous()).amax(-1, keepdim=True) * 0.125 * 68 * 2.0 ** -24
  p = s.softmax(-1)
  ref, size = p @ v, p @ v.abs()
  # the result's rounding, and errors of fp32 scores and sums: nothing of the size of a bf16 probability's
  assert bool(((out - ref).abs() <= ref.abs() * 2.0 ** -8 * 1.01 + size * (4 * off + 2.0 ** -18)).all())


def test_many_short_rows_of_own_keys():
  """Heads of 64 that share no keys, many and short: by the separate kernels, to the same result."""
  from types import SimpleNamespace
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  from xotorch_amd.models.llama import Attention
  from xotorch_amd.ops import torch_ref
  B, H, T, n = 128, 16, 100, 50
  cos, sin = torch_ref.rope_cos_sin(64, T, 10000.0, device="cuda")
  attn = Attention(SimpleNamespace(n_heads=H, n_kv_heads=H, head_dim=64, dim=64, attn_bias=False, qk_norm=False, norm_eps=1e-6))
  g = torch.Generator(device="cuda").manual_seed(0)
  rows = torch.randn(B, n, 3 * H * 64, generator=g, device="cuda").to(torch.bfloat16)
  qkv = torch.randn(B, 1, 3 * H * 64, generator=g, device="cuda").to(torch.bfloat16)
  at = torch.tensor([n], dtype=torch.int32, device="cuda")
  seen = torch.full((B,), n + 1, dtype=torch.int32, device="cuda")
  found = []
  for own in (True, False):
    c = ShardKVCache(1, B, H, T, 64, torch.bfloat16, "cuda")[0]
    ops.rope_qkv_append(rows.clone(), cos, sin, torch.arange(n, dtype=torch.int32, device="cuda"), c.k, c.v, H, H, 64, c.kp, c.vp)
    with torch.inference_mode():
      assert not ops.decode_attends(qkv, H, H, 64, c.kp) and ops.decode_attends(qkv[:127], H, H, 64, c.kp)
      if own:
        out = ops.decode_attend(qkv, cos, sin, at, seen, *c[:4], H, H)
      else:
        out = attn.attend(qkv.clone(), cos, sin, at, c, -1, True, seen)
    found.append((out, *c[:4]))
  for a, b in zip(found[0][1:], found[1][1:]):
    assert torch.equal(a, b)
  a, b = found[0][0].float(), found[1][0].float()
  assert bool(((a - b).abs() <= b.abs() * 2.0 ** -7 + 2.0 ** -14).all())  # both round fp32 sums in other orders


def test_lengths_of_more_rows_than_the_step_has():
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import ShardKVCache
  c = ShardKVCache(1, 3, 1, 32, 128, torch.bfloat16, "cuda")[0]
  g = torch.Generator(device="cuda").manual_seed(0)
  qkv = torch.randn(2, 1, 4 * 128, generator=g, device="cuda").to(torch.bfloat16)
  still, none = torch.ones(32, 64, device="cuda"), torch.zeros(32, 64, device="cuda")
  at = torch.zeros(2, dtype=torch.int32, device="cuda")
  seen = torch.ones(3, dtype=torch.int32, device="cuda")
  out = [ops.decode_attend(qkv, still, none, at, n, *c[:4], 2, 1) for n in (seen, seen[:2])]
  assert torch.equal(*out)
