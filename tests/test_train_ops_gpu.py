"""Differentiable operators of a training pass (hip/train_ops.hip) against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, STEP = torch.bfloat16, 2.0 ** -8  # what a result rounded to bf16 may be off by, of itself


def _rand(*shape, seed=0):
  g = torch.Generator(device="cuda").manual_seed(seed)
  return torch.randn(*shape, generator=g, device="cuda").to(BF)


def _norm64(f, w, add):
  return f * torch.rsqrt(f.square().mean(-1, keepdim=True) + 1e-5) * (w + add)


@pytest.mark.parametrize("rows,D", [(1, 8), (3, 2048), (700, 2056), (5, 4104), (2, 8200), (513, 64), (1, 16384)])
@pytest.mark.parametrize("residual", [False, True])
def test_norm(rows, D, residual):
  from xotorch_amd import ops
  x, r, w = _rand(2, rows, D), _rand(2, rows, D, seed=1), _rand(D, seed=2)
  dy, ds = _rand(2, rows, D, seed=3), _rand(2, rows, D, seed=4)
  leaves = [t.clone().requires_grad_(True) for t in (x, r, w)]
  exact = [t.double().requires_grad_(True) for t in (x, r, w)]
  if residual:
    y, s = ops.rmsnorm_residual(*leaves, 1e-5, 1.0)
    assert y.grad_fn is not None and "_NormResidual" in type(y.grad_fn).__name__
    torch.autograd.backward([y, s], [dy, ds])
    f = exact[0] + exact[1]
    torch.autograd.backward([_norm64(f, exact[2], 1.0), f], [dy.double(), ds.double()])
    assert torch.equal(leaves[0].grad, leaves[1].grad)
  else:
    y = ops.rmsnorm(leaves[0], leaves[2], 1e-5, 1.0)
    assert "_Norm" in type(y.grad_fn).__name__
    y.backward(dy)
    _norm64(exact[0], exact[2], 1.0).backward(dy.double())
    f = exact[0]
  f = f.detach()
  inv = torch.rsqrt(f.square().mean(-1, keepdim=True) + 1e-5)
  dn = dy.double() * (w.double() + 1)
  # fp32 sums over a row, scaled by the row
  terms = inv * (dn.abs() + f.abs() * inv * inv * (dn * f).abs().mean(-1, keepdim=True)) + (ds.double().abs() if residual else 0)
  ref = exact[0].grad
  assert bool(((leaves[0].grad.double() - ref).abs() <= ref.abs() * STEP + terms * (D + 16) * 2.0 ** -24).all())
  dw, size = exact[2].grad, (dy.double() * f * inv).abs().flatten(0, 1).sum(0)
  assert bool(((leaves[2].grad.double() - dw).abs() <= dw.abs() * STEP + size * (2 * rows + D) * 2.0 ** -24).all())


@pytest.mark.parametrize("rows,I", [(1, 8), (3, 1000), (257, 5632)])
def test_swiglu(rows, I):
  from xotorch_amd import ops
  gu, dy = (_rand(rows, 2 * I) * 4).requires_grad_(True), _rand(rows, I, seed=1)
  y = ops.swiglu_packed(gu)
  assert "_SwiGLU" in type(y.grad_fn).__name__
  y.backward(dy)
  e = gu.detach().double().requires_grad_(True)
  g, u = e.chunk(2, -1)
  (torch.nn.functional.silu(g) * u).backward(dy.double())
  # the sigmoid to a few 2^-22, in a sum with 1 that may cancel
  slack = (dy.double().abs() * (1 + g.abs() + u.abs() * (1 + g.abs()))).repeat(1, 2) * 2.0 ** -20
  assert bool(((gu.grad.double() - e.grad).abs() <= e.grad.abs() * STEP + slack).all())


@pytest.mark.parametrize("B,S,H,KVH,hd,per_row", [(1, 1, 1, 1, 8, False), (2, 33, 6, 2, 64, True), (2, 40, 4, 4, 128, False), (3, 5, 8, 1, 24, True)])
def test_heads(B, S, H, KVH, hd, per_row):
  from xotorch_amd.ops import torch_ref, train_ops
  cos, sin = torch_ref.rope_cos_sin(hd, 64, 10000.0, device="cuda")
  pos = torch.arange(3, 3 + S, dtype=torch.int32, device="cuda")
  pos = torch.stack([pos + b for b in range(B)]) if per_row else pos
  qkv = _rand(B, S, (H + 2 * KVH) * hd).requires_grad_(True)
  assert train_ops.takes_heads(qkv, cos, sin, pos, hd)
  out = train_ops._SplitHeads.apply(qkv, cos, sin, pos, H, KVH, hd)
  ref = train_ops._split(qkv.detach(), cos, sin, pos, H, KVH, hd)
  grads = [torch.randn(t.shape, device="cuda") for t in out]
  for a, b in zip(out, ref):  # x cos - y sin may be contracted differently: a step of bf16
    assert a.dtype == torch.float32 and a.is_contiguous() and bool(((a - b).abs() <= b.abs() * 2.0 ** -7 + 2.0 ** -20).all())
  torch.autograd.backward(out, grads)
  # exactly: the sum over heads that share a key, and the rotation's transpose
  dq, dk, dv = (g.double().view(B, -1, H // n, S, hd).sum(2).transpose(1, 2) for g, n in zip(grads, (H, KVH, KVH)))
  c, s = (t[pos.long()].double().expand(B, S, hd // 2)[:, :, None] for t in (cos, sin))
  def turned_back(g):
    g1, g2 = g.chunk(2, -1)
    return torch.cat([g1 * c + g2 * s, g2 * c - g1 * s], -1)
  ref = torch.cat([turned_back(dq), turned_back(dk), dv], 2).flatten(2)
  # rounded to bf16 before and after the turn; fp32 sums of H / KVH numbers
  size = torch.cat([dq, dk, dv], 2).abs()
  size = (size + size.roll(hd // 2, -1)).flatten(2)
  assert bool(((qkv.grad.double() - ref).abs() <= ref.abs() * STEP + size * (STEP + 2.0 ** -18)).all())
  o = torch.randn(B, H, S, hd, device="cuda").requires_grad_(True)
  m, d = train_ops._MergeHeads.apply(o), _rand(B, S, H * hd, seed=5)
  m.backward(d)
  assert torch.equal(m, o.detach().to(BF).transpose(1, 2).flatten(2)) and torch.equal(o.grad, d.view(B, S, H, hd).transpose(1, 2).float())


@pytest.mark.parametrize("B,S,H,KVH,hd,per_row", [(1, 1, 1, 1, 64, False), (2, 31, 6, 2, 64, True), (1, 33, 2, 2, 128, False),
                                                  (2, 200, 8, 1, 128, True), (1, 545, 4, 2, 64, False)])
@pytest.mark.parametrize("spread", [1.0, 4.0])
def test_causal_heads(B, S, H, KVH, hd, per_row, spread):
  from xotorch_amd.ops import torch_ref, train_ops
  cos, sin = torch_ref.rope_cos_sin(hd, 1024, 10000.0, device="cuda")
  pos = torch.arange(3, 3 + S, dtype=torch.int32, device="cuda")
  pos = torch.stack([pos + b for b in range(B)]) if per_row else pos
  qkv, d = (_rand(B, S, (H + 2 * KVH) * hd) * spread).requires_grad_(True), _rand(B, S, H * hd, seed=1)
  out = train_ops.causal_heads(qkv, cos, sin, pos, H, KVH, hd)
  assert "_CausalHeads" in type(out.grad_fn).__name__
  out.backward(d)
  # 64 bits from the rotated heads on (rounded to bf16, which the heads' test covers)
  q, k, v = (t.double().detach().requires_grad_(True) for t in train_ops._SplitHeads.apply(qkv.detach(), cos, sin, pos, H, KVH, hd))
  scores = (q @ k.transpose(-1, -2)) * hd ** -0.5
  p = scores.masked_fill(torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1), float("-inf")).softmax(-1)
  o, do = p @ v, d.view(B, S, H, hd).transpose(1, 2).double()
  o.backward(do)
  merged = o.detach().transpose(1, 2).flatten(2)
  # fp32 scores are off by their products' sizes, exponentials by as much relative to themselves
  with torch.no_grad():
    off = ((q.abs() @ k.abs().transpose(-1, -2)).amax(-1, keepdim=True) * hd ** -0.5 + 8) * (hd + 16) * 2.0 ** -24
    slack = (off * (p @ v.abs())).transpose(1, 2).flatten(2)
    assert bool(((out.double() - merged).abs() <= merged.abs() * STEP + slack).all())
    dp, delta = do.abs() @ v.abs().transpose(-1, -2), (do.abs() * (p @ v.abs())).sum(-1, keepdim=True)
    ds = p * (dp + delta) * (off + (hd + 16) * 2.0 ** -24) * hd ** -0.5
    slacks = [ds @ k.abs(), ds.transpose(-1, -2) @ q.abs(), (p * off).transpose(-1, -2) @ do.abs()]
    dq, dk, dv, sq, sk, sv = ((t.view(B, -1, H // n, S, hd).sum(2).transpose(1, 2))
                              for t, n in zip([q.grad, k.grad, v.grad] + slacks, (H, KVH, KVH) * 2))
    c, s = (t[pos.long()].double().expand(B, S, hd // 2)[:, :, None] for t in (cos, sin))
    def turned_back(g):
      g1, g2 = g.chunk(2, -1)
      return torch.cat([g1 * c + g2 * s, g2 * c - g1 * s], -1)
    ref = torch.cat([turned_back(dq), turned_back(dk), dv], 2).flatten(2)
    size, slack = torch.cat([dq, dk, dv], 2).abs(), torch.cat([sq, sk, sv], 2)
    size, slack = ((t + t.roll(hd // 2, -1)).flatten(2) for t in (size, slack))
    assert bool(((qkv.grad.double() - ref).abs() <= ref.abs() * STEP + size * (STEP + 2.0 ** -18) + slack).all())


@pytest.mark.parametrize("hd", [24, 64, 128])
def test_positions_as_torch_indexes(hd):
  """Negative ones count from the tables' end; past it there is nothing to train with."""
  from xotorch_amd.ops import torch_ref, train_ops
  B, S, H, KVH, T = 2, 40, 4, 2, 64
  cos, sin = torch_ref.rope_cos_sin(hd, T, 10000.0, device="cuda")
  at = torch.arange(T - S, T, dtype=torch.int32, device="cuda").expand(B, S).contiguous()
  d, found = _rand(B, S, H * hd, seed=1), []
  for pos in (at, at - T):
    qkv = _rand(B, S, (H + 2 * KVH) * hd).requires_grad_(True)
    assert train_ops.takes_heads(qkv, cos, sin, pos, hd)
    out = train_ops.causal_heads(qkv, cos, sin, pos, H, KVH, hd)
    out.backward(d)
    found.append((out, qkv.grad))
  assert all(torch.equal(a, b) for a, b in zip(*found))
  for bad in (T, -T - 1, 2 ** 31 - 1, -2 ** 31):
    pos = at.clone()
    pos[1, 33] = bad
    out = train_ops.causal_heads(_rand(B, S, (H + 2 * KVH) * hd).requires_grad_(True), cos, sin, pos, H, KVH, hd)
    assert torch.equal(out[0], found[0][0][0]) and bool(out[1, 33:].isnan().all())
    if hd != 24:  # (torch's attention spreads it to earlier tokens as well)
      assert torch.equal(out[1, :33], found[0][0][1, :33])
  short = torch.arange(T + 1, dtype=torch.int32, device="cuda")
  assert not train_ops.takes_heads(_rand(1, T + 1, (H + 2 * KVH) * hd).requires_grad_(True), cos, sin, short, hd)


@pytest.mark.parametrize("rows,K,N,rank,bias", [(1, 8, 24, 1, False), (5, 64, 40, 3, True), (130, 256, 520, 16, False),
                                                 (1, 256, 512, 1, False), (31, 512, 256, 4, True), (64, 768, 1280, 8, False),
                                                 (33, 256, 768, 11, True), (650, 2048, 256, 16, False)])
def test_adapted_linear(rows, K, N, rank, bias):
  from xotorch_amd.models.llama import XotLinear
  from xotorch_amd.train.lora import LoRALinear
  base = XotLinear(K, N, bias=bias).cuda().to(BF)
  lin = LoRALinear(base, rank=rank, alpha=3.0 * rank)
  with torch.no_grad():
    for n, p in enumerate(lin.parameters()):
      p.copy_(_rand(*p.shape, seed=10 + n) * 0.1)
  x, dy = _rand(2, rows, K).requires_grad_(True), _rand(2, rows, N, seed=1)
  y = lin(x)
  assert "_Adapted" in type(y.grad_fn).__name__ and y.shape == dy.shape
  assert ("_AdaptedRows" in type(y.grad_fn).__name__) == (K % 256 == N % 256 == 0)
  y.backward(dy)
  own = [y.detach(), x.grad, lin.lora_a.grad, lin.lora_b.grad]
  hook = base.register_forward_hook(lambda *_: None)  # somebody looks on: by separate operators
  x2 = x.detach().clone().requires_grad_(True)
  lin.lora_a.grad = lin.lora_b.grad = None
  y2 = lin(x2)
  assert "_Adapted" not in type(y2.grad_fn).__name__
  y2.backward(dy)
  hook.remove()
  base.forward = lambda t: XotLinear.forward(base, t)  # or put something in its place
  assert "_Adapted" not in type(lin(x2).grad_fn).__name__
  del base.forward
  w, a, b, e, d = (t.detach().double() for t in (base.weight, lin.lora_a.to(BF), lin.lora_b.to(BF), x.flatten(0, 1), dy.flatten(0, 1)))
  low, dlow = e @ a.t(), 3.0 * d @ b
  ref = [e @ w.t() + (base.bias.double() if bias else 0) + 3 * low @ b.t(), d @ w + dlow @ a, dlow.t() @ e, 3 * d.t() @ low]
  size = [e.abs() @ w.abs().t() + 1 + 3 * (e.abs() @ a.abs().t()) @ b.abs().t(), d.abs() @ w.abs() + 3 * (d.abs() @ b.abs()) @ a.abs(),
          3 * (d.abs() @ b.abs()).t() @ e.abs(), 3 * d.abs().t() @ (e.abs() @ a.abs().t())]
  for o, o2, r, z in zip(own, [y2.detach(), x2.grad, lin.lora_a.grad, lin.lora_b.grad], ref, size):
    # a result and its low-rank factor are rounded to bf16, as without the function
    assert bool(((o.double().view(r.shape) - r).abs() <= r.abs() * 2 * STEP + z * STEP).all())
    assert (o.double().view(r.shape) - r).norm() <= 1.1 * (o2.double().view(r.shape) - r).norm() + 1e-3 * r.norm()
  twice = torch.autograd.grad(lin(x), x, dy, create_graph=True)[0]
  twice.float().square().sum().backward()
  both = torch.autograd.grad(lin(x), (x, lin.lora_a, lin.lora_b), torch.stack([dy, dy]), is_grads_batched=True)
  for o, r, z in zip(both, ref[1:], size[1:]):
    assert bool(((o[1].double().view(r.shape) - r).abs() <= r.abs() * 2 * STEP + z * STEP).all())


@pytest.mark.parametrize("rank", [1, 5, 16])
@pytest.mark.parametrize("M", [1, 63, 64, 65, 129, 1500])
def test_narrow_sums(M, rank):
  """Rows and columns at the edges of steps; what lies past a tensor's rows counts nowhere."""
  from xotorch_amd.ops import train_ops
  hip, N = train_ops._hip_lora(), 768
  t, w, c = _rand(M, N), _rand(N, rank, seed=2).float() * 1.001, _rand(16, -(-M // 64) * 64, seed=3)
  c[rank:], c[:, M:] = 0, 0
  wt = w.t().contiguous()
  low, lowt, down = hip.sums(t, wt, 0.5, c, rank, 3.0, False)
  again, _ = hip.sums(t, wt, 0.5, None, rank, 1.0, False)
  turned, = hip.sums(t, None, 1.0, c, rank, 3.0, True)
  assert torch.equal(low, again) and torch.equal(turned.t(), down) and down.shape == (N, rank)
  td, wd, cd = t.double(), w.to(BF).double(), c[:rank, :M].double()
  rows, cols = 0.5 * td @ wd, 3.0 * td.t() @ cd.t()
  assert bool(((low[:, :rank].double() - rows).abs() <= (td.abs() @ wd.abs()) * (N + 8) * 2.0 ** -25).all()) and not low[:, rank:].any()
  assert bool(((down.double() - cols).abs() <= (td.abs().t() @ cd.abs().t()) * (M + 8) * 3 * 2.0 ** -24).all())
  assert torch.equal(lowt[:rank, :M], low[:, :rank].t().to(BF)) and not lowt[rank:].any() and not lowt[:, M:].any()
  out, by = _rand(M, N, seed=4), low[:, :rank].double() @ (2.0 * w.double().t())
  want = out.double() + by
  hip.add(out, low, wt, 2.0)
  slack = (low[:, :rank].double().abs() @ (2.0 * w.double().abs().t()) + want.abs()) * (rank + 4) * 2.0 ** -24
  assert bool(((out.double() - want).abs() <= slack + want.abs() * 2.0 ** -8).all())
  t[M - 1, 5] = float("inf")
  low, _, down = hip.sums(t, wt, 1.0, c, rank, 1.0, False)
  assert low[:M - 1].isfinite().all() and torch.equal(down.isnan(), (t.float().t() @ c[:rank, :M].float().t()).isnan())


@pytest.mark.parametrize("rank", [1, 3, 4, 5, 12])
def test_narrow_sums_of_infinities(rank):
  """Features that fill a rank up add nothing: a row that holds an infinity is one, and not a number,
  where fp32 says so."""
  from xotorch_amd.ops import train_ops
  hip, M, N = train_ops._hip_lora(), 70, 512
  t, w, out = _rand(M, N), _rand(rank, N, seed=2).float(), _rand(M, N, seed=3)
  t[33, 5], t[M - 1, 300] = float("inf"), -float("inf")
  low, lowt = hip.sums(t, w, 1.0, None, rank, 1.0, False)
  assert not low[:, rank:].any() and not lowt[rank:].any()
  want = out.float() + sum(low[:, r:r + 1] * w[r] for r in range(rank))
  hip.add(out, low, w, 1.0)
  assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())


def test_second_derivatives_forward_mode_and_transforms():
  """What the functions cannot do themselves goes by torch's operators."""
  from xotorch_amd import ops
  from xotorch_amd.ops import torch_ref
  x, w, gu, dy = _rand(3, 64), _rand(64, seed=1), _rand(3, 128, seed=2), _rand(3, 64, seed=3)
  for own, ref, at in ((lambda t: ops.rmsnorm(t, w, 1e-5), lambda t: torch_ref.rmsnorm(t, w, 1e-5), x),
                       (lambda t: ops.rmsnorm_residual(t, dy, w, 1e-5)[0], lambda t: torch_ref.rmsnorm_residual(t, dy, w, 1e-5)[0], x),
                       (ops.swiglu_packed, torch_ref.swiglu_packed, gu)):
    found = []
    for f in (own, ref):
      t = at.clone().requires_grad_(True)
      g, = torch.autograd.grad(f(t), t, dy, create_graph=True)
      found.append(torch.autograd.grad(g.float().square().sum(), t)[0].float())
    assert (found[0] - found[1]).norm() <= 0.02 * found[1].norm()  # bf16 gradients of bf16 gradients
    assert torch.equal(torch.func.vmap(torch.func.grad(lambda t: own(t).float().sum()))(at[:, None]),
                       torch.func.vmap(torch.func.grad(lambda t: ref(t).float().sum()))(at[:, None]))
    t = at.clone().requires_grad_(True)
    with torch.autograd.forward_ad.dual_level():
      dual = torch.autograd.forward_ad.make_dual(t, torch.ones_like(t))
      assert torch.autograd.forward_ad.unpack_dual(own(dual)).tangent is not None
