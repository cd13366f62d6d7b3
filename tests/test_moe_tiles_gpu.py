"""Prompts through routed experts by tiles against a loop over experts in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,D,I", [(257, 8, 2, 128, 192), (300, 3, 2, 64, 64), (1500, 8, 2, 192, 320), (700, 16, 1, 64, 128),
                                       (2000, 5, 4, 256, 448)])
def test_prompt_by_tiles(T, E, k, D, I):
  from xotorch_amd.models.config import ModelConfig
  from xotorch_amd.models.llama import MoEMLP
  g = torch.Generator(device="cuda").manual_seed(T)
  moe = MoEMLP(ModelConfig(dim=D, n_experts=E, n_experts_per_tok=k, intermediate_dim=I)).to("cuda", torch.bfloat16)
  x = torch.randn(1, T, D, generator=g, device="cuda").to(torch.bfloat16)
  with torch.no_grad():
    for p in moe.parameters():
      p.copy_(torch.randn(p.shape, generator=g, device="cuda") * p.shape[-1] ** -0.5)
    moe.gate.weight.mul_(4)  # decided choices: the best of the rest is rarely within rounding
    assert moe._grouped(x[0]) is not None and moe._many(x[0])
    out = moe(x)[0].double()
    xd = x[0].double()
    logits = xd @ moe.gate.weight.double().t()
    w, chosen = logits.softmax(-1).topk(k)
    w = w / w.sum(-1, keepdim=True)
    ref, size = torch.zeros_like(xd), torch.zeros_like(xd)
    for e in range(E):
      token, place = torch.where(chosen == e)
      gate, up = (xd[token] @ moe.experts[e].gate_up_proj.weight.double().t()).chunk(2, -1)
      h = torch.nn.functional.silu(gate) * up
      down = moe.experts[e].down_proj.weight.double()
      ref.index_add_(0, token, h @ down.t() * w[token, place, None])
      size.index_add_(0, token, h.abs() @ down.abs().t() * w[token, place, None])
    # activations, rows and the sum are bf16 once each; the rest is fp32
    near = logits.topk(min(k + 1, E)).values
    sure = (near[:, k - 1] - near[:, -1] > 1e-4) if E > k else torch.ones(T, dtype=torch.bool, device="cuda")
    assert sure.float().mean() > 0.99
    bound = size * 2.0 ** -7 + ref.abs() * 2.0 ** -8 + 1e-6
    assert bool(((out - ref).abs() <= bound)[sure].all())


@pytest.mark.parametrize("T,E,k,D", [(1, 8, 2, 64), (33, 5, 3, 72), (256, 128, 8, 128)])
def test_routes_of_bf16_logits_and_wide_sums(T, E, k, D):
  """bf16 logits go as the same numbers in fp32 do; a wide sum is one that is not rounded yet."""
  from xotorch_amd import ops
  hip = ops._load_hip()
  g = torch.Generator(device="cuda").manual_seed(T)
  logits = torch.randn(T, E, generator=g, device="cuda").to(torch.bfloat16)
  (idx, w), (idx2, w2) = hip.moe_route(logits, None, k, 0), hip.moe_route(logits.float(), None, k, 0)
  assert torch.equal(idx, idx2) and torch.equal(w, w2)
  gather, place = hip.moe_build(idx, E, (T + 31) // 32 * 32)
  y = torch.randn(gather.numel(), D, generator=g, device="cuda").to(torch.bfloat16)
  wide, rounded = hip.moe_combine(y, place, w, True), hip.moe_combine(y, place, w)
  assert wide.dtype == torch.float32 and torch.equal(wide.to(torch.bfloat16), rounded)


@pytest.mark.parametrize("E,k,mode,groups,keep", [(8, 2, 0, 1, 1), (5, 5, 0, 1, 1), (256, 8, 0, 1, 1), (16, 4, 1, 1, 1), (16, 6, 1, 4, 1)])
def test_every_pick_is_another_expert(E, k, mode, groups, keep):
  """Rows that are no numbers, infinities and fewer open experts than picks: a token has one row in an expert,
  which is what the room for its rows is made for."""
  from xotorch_amd import ops
  hip = ops._load_hip()
  T = 33
  g = torch.Generator(device="cuda").manual_seed(E)
  logits = torch.randn(T, E, generator=g, device="cuda")
  logits[3], logits[4], logits[5] = torch.nan, torch.inf, -torch.inf
  logits[6, 1], logits[7, E - 1] = torch.nan, torch.inf
  logits[8, 1:] = -torch.inf  # one expert is open
  for given in (logits, logits.to(torch.bfloat16)):
    idx, w = hip.moe_route(given, None, k, mode, groups, keep)
    at = idx.long().sort(-1).values
    assert int(at.min()) >= 0 and int(at.max()) < E and bool((at.diff(dim=-1) > 0).all())
    assert bool(w[3].isnan().all()) and bool(w[9:].isfinite().all())
    if mode == 0:
      assert bool(w[6].isnan().all()) and float(w[8].max()) == 1.0 and int(idx[8, 0]) == 0
    C = 64
    gather, place = hip.moe_build(idx, E, C)
    assert bool((place.long() // C == idx).all()) and place.unique().numel() == T * k and bool((gather[place.long()] == torch.arange(T, device="cuda")[:, None]).all())


@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("K,F", [(64, 16), (128, 144), (192, 272), (320, 64), (576, 528)])  # steps of k, tiles of features
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("few", [False, True])  # on average up to 56 rows an expert, or more
def test_rows_of_an_expert(tile, K, F, swiglu, few):
  """Experts of all numbers of rows at which a tile's form changes, none among them."""
  from xotorch_amd.ops.mixer_ops import load_hip
  hip = load_hip("_hip_experts")
  counts = [0, 1, 64, 0, 65, 129] if few else [0, 63, 128, 129, 0, 192, 193, 256, 257, 321, 513, 700, 1]
  assert (sum(counts) <= 56 * len(counts)) == few
  first = [0]
  for c in counts:
    first.append(first[-1] + c)
  pairs = first[-1]
  tiles = [(e, r) for e in range(len(counts)) for r in range(first[e], first[e + 1], tile)]
  most = pairs // tile + len(counts)
  listed = tiles + [(-1, 0)] * (most - len(tiles)) + [(-1, len(tiles))]
  g = torch.Generator(device="cuda").manual_seed(K + F)
  n = pairs // 2 + 1
  x = torch.randn(n if swiglu else pairs, K, generator=g, device="cuda").to(torch.bfloat16)
  token = torch.randint(0, n, (pairs,), generator=g, device="cuda", dtype=torch.int32)
  w = [(torch.randn((2 if swiglu else 1) * F, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16) for _ in counts]
  ints = dict(dtype=torch.int32, device="cuda")
  got = hip.expert_product_of(x, w, token, torch.tensor(first, **ints), torch.tensor(listed, **ints), tile, swiglu)
  rows = (x[token.long()] if swiglu else x).double()
  for e in range(len(counts)):
    r = rows[first[e]:first[e + 1]]
    want, size = r @ w[e].double().t(), r.abs() @ w[e].double().abs().t()
    slack = size * (K + 8) * 2.0 ** -24  # fp32 sums of K products
    if swiglu:
      (gate, up), (sg, su) = want.chunk(2, -1), slack.chunk(2, -1)
      want = torch.nn.functional.silu(gate) * up
      # silu's slope is at most 1.1; its hardware exponential and reciprocal are off by some 2^-20
      slack = (1.1 * sg + gate.abs() * 2.0 ** -19) * up.abs() + su * gate.abs()
    assert bool(((got[first[e]:first[e + 1]].double() - want).abs() <= slack + want.abs() * 2.0 ** -8 + 1e-30).all()), counts[e]


@pytest.mark.parametrize("rows", [[129, 160, 161, 224, 225], [150, 0, 200, 300, 450, 33], [96, 97, 320, 321, 447, 448]])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("F", [528, 3600])  # few blocks, whose tiles the kernel plans, and the router's tiles
def test_shares_of_rows_in_steps_of_32(rows, swiglu, F):
  """Tiles of 160 and 224 rows, whole and cut in two: what one row gives does not depend on its tile's form."""
  from xotorch_amd.ops.mixer_ops import load_hip
  hip = load_hip("_hip_experts")
  K, n = 320, sum(rows)
  g = torch.Generator(device="cuda").manual_seed(n)
  x = torch.randn(n, K, generator=g, device="cuda").to(torch.bfloat16)
  w = [(torch.randn((2 if swiglu else 1) * F, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16) for _ in rows]
  ints = dict(dtype=torch.int32, device="cuda")

  def product(counts, some, weights, tile):
    first = [0]
    for c in counts:
      first.append(first[-1] + c)
    tiles = [(e, r) for e in range(len(counts)) for r in range(first[e], first[e + 1], tile)]
    most = first[-1] // tile + len(counts)
    listed = tiles + [(-1, 0)] * (most - len(tiles)) + [(-1, len(tiles))]
    token = torch.arange(first[-1], **ints)
    return hip.expert_product_of(some, weights, token, torch.tensor(first, **ints), torch.tensor(listed, **ints), tile, swiglu), first

  got, first = product(rows, x, w, 256)
  for e, c in enumerate(rows):
    if c:
      alone = product([c], x[first[e]:first[e + 1]].contiguous(), [w[e]], 128)[0]
      assert torch.equal(got[first[e]:first[e + 1]], alone)
      some, weights = x[first[e]:first[e + 1]].double(), w[e].double()
      want, size = some @ weights.t(), some.abs() @ weights.abs().t() * (K + 8) * 2.0 ** -24  # fp32 sums of K products
      if swiglu:
        (gate, up), (sg, su) = want.chunk(2, -1), size.chunk(2, -1)
        want = torch.nn.functional.silu(gate) * up
        # silu's slope is at most 1.1; its hardware exponential and reciprocal are off by some 2^-20
        size = (1.1 * sg + gate.abs() * 2.0 ** -19) * (up.abs() + su) + su * gate.abs()
      assert bool(((got[first[e]:first[e + 1]].double() - want).abs() <= size + want.abs() * 2.0 ** -8 + 1e-30).all()), c


@pytest.mark.parametrize("experts,F", [(1, 2048), (8, 4096), (65, 272), (130, 48), (250, 16)])  # one, some or many a lane
def test_tiles_that_the_kernel_plans(experts, F, K=64):
  """Few rounds of blocks: whatever rows a tile has, each row is what its expert gives it alone."""
  from xotorch_amd.ops.mixer_ops import load_hip
  hip = load_hip("_hip_experts")
  g = torch.Generator(device="cuda").manual_seed(experts)
  sizes = [0, 1, 100, 128, 129, 190, 193, 256, 257, 300, 384, 385]
  w = [(torch.randn(F, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16) for _ in range(experts)]
  ints = dict(dtype=torch.int32, device="cuda")
  for spread in range(4):
    if spread == 3: counts = [sizes[(5 * e) % len(sizes)] for e in range(experts)]
    else: counts = [(260, 390, 150)[spread] + e % 3 for e in range(experts)]
    first = [0]
    for c in counts:
      first.append(first[-1] + c)
    pairs = first[-1]
    if pairs == 0: continue
    x = torch.randn(pairs, K, generator=g, device="cuda").to(torch.bfloat16)
    tiles = [(e, r) for e in range(experts) for r in range(first[e], first[e + 1], 256)]
    listed = tiles + [(-1, 0)] * (pairs // 256 + experts - len(tiles)) + [(-1, len(tiles))]
    got = hip.expert_product_of(x, w, torch.arange(pairs, **ints), torch.tensor(first, **ints), torch.tensor(listed, **ints), 256, False)
    for e in range(experts):
      rows = x[first[e]:first[e + 1]].double()
      want, size = rows @ w[e].double().t(), rows.abs() @ w[e].double().abs().t()
      slack = size * (K + 8) * 2.0 ** -24 + want.abs() * 2.0 ** -8 + 1e-30  # fp32 sums of K products
      assert bool(((got[first[e]:first[e + 1]].double() - want).abs() <= slack).all()), (spread, e, counts[e])


@pytest.mark.parametrize("experts,F", [(8, 4096), (65, 272), (130, 48), (250, 16)])
def test_more_tiles_that_the_kernel_plans(experts, F):
  """As many blocks as it plans of long rows only"""
  test_tiles_that_the_kernel_plans(experts, F, 4224)


def test_tokens_past_four_gigabytes():
  """Offsets of more than 32 bits, of the last tokens of all."""
  from xotorch_amd.ops.mixer_ops import load_hip
  hip = load_hip("_hip_experts")
  T, K, F, n = (1 << 20) + 40, 2048, 32, 300
  x = torch.zeros(T, K, device="cuda", dtype=torch.bfloat16)
  g = torch.Generator(device="cuda").manual_seed(T)
  token = torch.cat([torch.randint(0, T, (n - 2,), generator=g, device="cuda"), torch.tensor([0, T - 1], device="cuda")])
  x[token] = torch.randn(n, K, generator=g, device="cuda").to(torch.bfloat16)
  w = (torch.randn(2 * F, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
  ints = dict(dtype=torch.int32, device="cuda")
  for tile in (128, 256):
    tiles = [(0, r) for r in range(0, n, tile)]
    listed = tiles + [(-1, 0)] * (n // tile + 1 - len(tiles)) + [(-1, len(tiles))]
    args = torch.tensor([0, n], **ints), torch.tensor(listed, **ints), tile, True
    near = hip.expert_product_of(x[token].contiguous(), [w], torch.arange(n, **ints), *args)
    assert torch.equal(hip.expert_product_of(x, [w], token.to(torch.int32), *args), near)


@pytest.mark.parametrize("kind", ["GATED", "RELU2"])
@pytest.mark.parametrize("tile,F", [(128, 32), (128, 33024), (256, 32)])  # half blocks, whole ones, large tiles
def test_stacked_weights_of_tokens_past_four_gigabytes(kind, tile, F):
  """The same with rows that end within a step."""
  from xotorch_amd.ops.mixer_ops import load_hip
  hip = load_hip("_hip_experts")
  T, K, kp, n = (1 << 20) + 40, 2056, 2112, 300
  x = torch.zeros(T, K, device="cuda", dtype=torch.bfloat16)
  g = torch.Generator(device="cuda").manual_seed(T)
  token = torch.cat([torch.randint(0, T, (n - 2,), generator=g, device="cuda"), torch.tensor([0, T - 1], device="cuda")])
  x[token] = torch.randn(n, K, generator=g, device="cuda").to(torch.bfloat16)
  F = F if kind == "RELU2" else max(16, F // 32 * 16)
  w = torch.zeros(*((1, 2, F, kp) if kind == "GATED" else (1, F, kp)), device="cuda", dtype=torch.bfloat16)
  w[..., :K] = (torch.randn(*w.shape[:-1], K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
  ints = dict(dtype=torch.int32, device="cuda")
  tiles = [(0, r) for r in range(0, n, tile)]
  listed = tiles + [(-1, 0)] * (n // tile + 1 - len(tiles)) + [(-1, len(tiles))]
  args = torch.tensor([0, n], **ints), torch.tensor(listed, **ints), tile, getattr(hip, kind), 1.0, 100.0, 0.0
  near = hip.expert_product(x[token].contiguous(), w, torch.arange(n, **ints), *args)
  assert torch.equal(hip.expert_product(x, w, token.to(torch.int32), *args), near) and bool(near.any())


@pytest.mark.parametrize("swiglu", [False, True])
def test_rows_past_what_tiles_address(swiglu):
  from xotorch_amd.ops.mixer_ops import load_hip
  hip = load_hip("_hip_experts")
  K, F, counts = (1 << 22) + 64, 16, [17, 0, 3]
  g, n = torch.Generator(device="cuda").manual_seed(K), sum(counts)
  x = torch.randn(n, K, generator=g, device="cuda", dtype=torch.bfloat16)
  w = [torch.randn((2 if swiglu else 1) * F, K, generator=g, device="cuda", dtype=torch.bfloat16) * 2.0 ** -11 for _ in counts]
  ints = dict(dtype=torch.int32, device="cuda")
  first, tiles = torch.tensor([0, 17, 17, 20], **ints), torch.tensor([(0, 0), (2, 17), (-1, 0), (-1, 2)], **ints)
  got = hip.expert_product_of(x, w, torch.arange(n, **ints), first, tiles, 128, swiglu).double()
  for e, (lo, hi) in ((0, (0, 17)), (2, (17, 20))):
    want = x[lo:hi].double() @ w[e].double().t()
    # fp32 sums by four waves, each of K / 128 additions of 32 products; of random signs, they stay
    # within six standard deviations
    slack = x[lo:hi].double().norm(dim=1, keepdim=True) * w[e].double().norm(dim=1) * K ** -0.5 * 6 * (K / 128 + 8) * 2.0 ** -24
    if swiglu:
      (gate, up), (sg, su) = want.chunk(2, -1), slack.chunk(2, -1)
      want = torch.nn.functional.silu(gate) * up
      slack = (1.1 * sg + gate.abs() * 2.0 ** -19) * (up.abs() + su) + su * gate.abs()
    assert bool(((got[lo:hi] - want).abs() <= slack + want.abs() * 2.0 ** -8).all()), e


@pytest.mark.parametrize("K,F", [(64, 16), (192, 272), (320, 48), (2048, 80)])  # 1, 3, 5 and 32 steps, the last begun at different places
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("counts", [[0, 1, 16, 17, 0, 2], [33, 64, 65, 0, 128, 129, 200, 1, 32], [3]])  # 64 weight rows a block, and 128
def test_few_rows_of_an_expert(K, F, swiglu, counts):
  from xotorch_amd.ops.mixer_ops import load_hip
  hip = load_hip("_hip_experts")
  first = [0]
  for c in counts:
    first.append(first[-1] + c)
  pairs = first[-1]
  tiles = [(e, r) for e in range(len(counts)) for r in range(first[e], first[e + 1], 128)]
  listed = tiles + [(-1, 0)] * (pairs // 128 + len(counts) - len(tiles)) + [(-1, len(tiles))]
  g = torch.Generator(device="cuda").manual_seed(K + F)
  n = pairs // 2 + 1
  x = torch.randn(n if swiglu else pairs, K, generator=g, device="cuda").to(torch.bfloat16)
  token = torch.randint(0, n, (pairs,), generator=g, device="cuda", dtype=torch.int32)
  w = [(torch.randn((2 if swiglu else 1) * F, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16) for _ in counts]
  ints = dict(dtype=torch.int32, device="cuda")
  places = token, torch.tensor(first, **ints), torch.tensor(listed, **ints), 128
  got = hip.expert_few_of(x, w, *places, swiglu)
  rows = (x[token.long()] if swiglu else x).double()
  for e in range(len(counts)):
    r = rows[first[e]:first[e + 1]]
    want, size = r @ w[e].double().t(), r.abs() @ w[e].double().abs().t()
    slack = size * (K + 8) * 2.0 ** -24  # as above
    if swiglu:
      (gate, up), (sg, su) = want.chunk(2, -1), slack.chunk(2, -1)
      want = torch.nn.functional.silu(gate) * up
      slack = (1.1 * sg + gate.abs() * 2.0 ** -19) * (up.abs() + su) + su * gate.abs()
    assert bool(((got[first[e]:first[e + 1]].double() - want).abs() <= slack + want.abs() * 2.0 ** -8 + 1e-30).all()), counts[e]


@pytest.mark.parametrize("T,E,k,D,I", [(1, 8, 2, 64, 128), (16, 8, 2, 128, 64), (17, 5, 3, 192, 64), (200, 128, 8, 128, 192), (256, 16, 2, 64, 64),
                                       (300, 64, 4, 64, 64)])
def test_few_tokens_through_experts(T, E, k, D, I):
  """Router blocks of 16 tokens whose counts need no scan, and more of them; rows left as they are for a wide sum."""
  from xotorch_amd.models.config import ModelConfig
  from xotorch_amd.models.llama import MoEMLP
  g = torch.Generator(device="cuda").manual_seed(T)
  moe = MoEMLP(ModelConfig(dim=D, n_experts=E, n_experts_per_tok=k, intermediate_dim=I)).to("cuda", torch.bfloat16)
  x = torch.randn(T, D, generator=g, device="cuda").to(torch.bfloat16)
  with torch.no_grad():
    for p in moe.parameters():
      p.copy_(torch.randn(p.shape, generator=g, device="cuda") * p.shape[-1] ** -0.5)
    moe.gate.weight.mul_(4)
    assert moe._grouped(x) is not None and not moe._many(x)
    out, wide = moe(x[None])[0], moe._forward_decode(x, True)
    assert wide.dtype == torch.float32 and torch.equal(wide.to(torch.bfloat16), out)
    xd = x.double()
    logits = xd @ moe.gate.weight.double().t()
    w, chosen = logits.softmax(-1).topk(k)
    w = w / w.sum(-1, keepdim=True)
    ref, size = torch.zeros_like(xd), torch.zeros_like(xd)
    for e in range(E):
      token, place = torch.where(chosen == e)
      gate, up = (xd[token] @ moe.experts[e].gate_up_proj.weight.double().t()).chunk(2, -1)
      h = torch.nn.functional.silu(gate) * up
      down = moe.experts[e].down_proj.weight.double()
      ref.index_add_(0, token, h @ down.t() * w[token, place, None])
      size.index_add_(0, token, h.abs() @ down.abs().t() * w[token, place, None])
    # up to 256 tokens logits are bf16, each off by 2^-9 of it: a choice by less than two of these may be another, and
    # a weight is off by as much, of itself
    loose = logits.abs().amax(-1) * 2.0 ** -8 if T <= 256 else torch.zeros(T, dtype=torch.float64, device="cuda")
    near = logits.topk(min(k + 1, E)).values
    sure = near[:, k - 1] - near[:, -1] > 1e-4 + loose
    assert sure.float().mean() > 0.8
    # activations, rows and the sum are bf16 once each; the rest is fp32
    assert bool(((out.double() - ref).abs() <= size * (2.0 ** -7 + 1.01 * loose[:, None]) + ref.abs() * 2.0 ** -8 + 1e-6)[sure].all())
    # someone who waits for an expert gets its call
    seen = []
    moe.experts[0].register_forward_hook(lambda *a: seen.append(1))
    assert moe._grouped(x) is None


@pytest.mark.parametrize("mode", ["auto", "all"])
def test_no_copies_of_experts_that_are_read_where_they_lie(mode, monkeypatch):
  from xotorch_amd.models.config import config_from_hf
  from xotorch_amd.models.llama import ShardedModel
  from xotorch_amd.models.registry import builtin_config
  from xotorch_amd.shard import Shard
  raw = dict(builtin_config("mixtral-8x7b"))
  raw.update(hidden_size=256, intermediate_size=512, num_attention_heads=4, num_key_value_heads=2, vocab_size=256)
  cfg = config_from_hf(raw, "mixtral-gpu-tiny")
  model = ShardedModel(cfg, Shard("mixtral-gpu-tiny", 1, 1, cfg.n_layers)).to("cuda", torch.bfloat16)
  monkeypatch.setenv("XOT_PACK", mode)
  model.pack_decode_weights()
  layer = model.layers["1"]
  assert layer.mlp.wp_gate_up is None and all(p.weight_packed is None for e in layer.mlp.experts for p in (e.gate_up_proj, e.down_proj))
  assert (layer.self_attn.o_proj.weight_packed is not None) == (mode == "all")
  # an expert with a hook has its call, which may read a copy
  layer.mlp.experts[2].register_forward_hook(lambda *a: None)
  model.pack_decode_weights()
  assert layer.mlp.wp_gate_up is not None


@pytest.mark.parametrize("T", [257, 300, 500])
def test_prompts_beside_fp8_copies(T, monkeypatch):
  """Copies for decode leave prompts to the grouped products, which read the weights themselves."""
  from xotorch_amd.models.config import ModelConfig
  from xotorch_amd.models.llama import MoEMLP
  g = torch.Generator(device="cuda").manual_seed(T)
  moe = MoEMLP(ModelConfig(dim=256, n_experts=32, n_experts_per_tok=2, intermediate_dim=128)).to("cuda", torch.bfloat16)
  x = torch.randn(1, T, 256, generator=g, device="cuda").to(torch.bfloat16)
  with torch.no_grad():
    for p in moe.parameters():
      p.copy_(torch.randn(p.shape, generator=g, device="cuda") * p.shape[-1] ** -0.5)
    want = moe(x)
    monkeypatch.setenv("XOT_FP8_GEMM", "1")
    for e in moe.experts:
      e.gate_up_proj.pack_decode()
      e.down_proj.pack_decode()
    moe.pack_grouped()
    assert moe.wp_gate_up_fp8 is not None
    assert moe._grouped(x[0]) is not None and moe._grouped(x[0, :256]) is None
    assert torch.equal(moe(x), want)
    monkeypatch.setenv("XOT_FP8_PREFILL", "1")
    assert moe._grouped(x[0]) is None


@pytest.mark.parametrize("T", [1, 40, 256])
@pytest.mark.parametrize("who", ["hook", "global hook", "autocast", "dispatch mode", "module of its own", "bias"])
def test_experts_of_a_router_with_its_own_call(T, who):
  """A router that somebody waits for is called, and its experts still go as two grouped products: the same numbers, as
  whole ones are summed and rounded alike by either way. More tokens have all modules called."""
  import contextlib
  from torch.utils._python_dispatch import TorchDispatchMode
  from xotorch_amd.models.config import ModelConfig
  from xotorch_amd.models.llama import MoEMLP

  class Seen(TorchDispatchMode):
    def __torch_dispatch__(self, f, types, args=(), kwargs=None):
      return f(*args, **(kwargs or {}))

  class Router(torch.nn.Linear):
    pass

  E, k, D, I = 16, 4, 128, 192
  g = torch.Generator(device="cuda").manual_seed(T)
  moe = MoEMLP(ModelConfig(dim=D, n_experts=E, n_experts_per_tok=k, intermediate_dim=I)).to("cuda", torch.bfloat16)
  make = lambda n: torch.randint(-1, 2, (n, D), generator=g, device="cuda").to(torch.bfloat16)
  x, more = make(T), make(300)
  with torch.no_grad():
    for p in moe.parameters():
      p.copy_(torch.randn(p.shape, generator=g, device="cuda") * p.shape[-1] ** -0.5)
    moe.gate.weight.copy_(make(E))  # logits are whole numbers of up to 128
    want, many = moe(x[None]), moe(more[None])
    if who == "bias":  # whole numbers too, which the experts' call has to see
      from torch.nn.functional import linear
      bias = torch.randint(-9, 10, (E,), generator=g, device="cuda").to(torch.bfloat16)
      direct = moe.gate.weight
      moe.gate = torch.nn.Linear(D, E, device="cuda", dtype=torch.bfloat16)
      moe.gate.weight, moe.gate.bias = direct, torch.nn.Parameter(bias)
      found = moe._grouped(x)
      assert found is not None and found[2] is None and moe._grouped(more) is None
      w, chosen = linear(x.double(), direct.double(), bias.double()).softmax(-1).topk(k)
      w, ref = w / w.sum(-1, keepdim=True), torch.zeros(T, D, dtype=torch.float64, device="cuda")
      for e in range(E):
        token, place = torch.where(chosen == e)
        gate, up = (x.double()[token] @ moe.experts[e].gate_up_proj.weight.double().t()).chunk(2, -1)
        h = torch.nn.functional.silu(gate) * up
        ref.index_add_(0, token, h @ moe.experts[e].down_proj.weight.double().t() * w[token, place, None])
      off = (moe(x[None])[0].double() - ref).norm(dim=-1) / ref.norm(dim=-1)
      assert float(off.median()) < 1e-2  # tokens with equal logits may choose otherwise
      return
    if who == "module of its own":
      router = Router(D, E, bias=False)
      router.weight = moe.gate.weight
      moe.gate = router
    called = []
    with contextlib.ExitStack() as s:
      if who in ("hook", "module of its own"):
        h = moe.gate.register_forward_hook(lambda m, *a: called.append(m))
      else:
        h = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: called.append(m))
      s.callback(h.remove)
      if who == "autocast":
        s.enter_context(torch.autocast("cuda", torch.bfloat16))
      if who == "dispatch mode":
        s.enter_context(Seen())
      found = moe._grouped(x)
      assert found is not None and found[2] is None and moe._grouped(more) is None
      got = moe(x[None])
      assert [m for m in called if m is not moe] == [moe.gate]
      assert torch.equal(got, want)
      after = moe(more[None])
      assert who in ("hook", "module of its own") or len(called) > 2 * k
    assert (after.float() - many.float()).norm() <= 0.02 * many.float().norm()
    assert moe._forward_decode(x, True).dtype == torch.float32
