"""Which calls go to the kernels: those that can read their operands and that nobody follows."""
import random

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

BF = torch.bfloat16


def test_fake_tensors_are_not_read_in_training():
  from xotorch_amd.models.llama import XotLinear
  from xotorch_amd.ops import train_ops
  from xotorch_amd.train.lora import LoRALinear
  with FakeTensorMode():
    x = torch.empty(2, 3, 512, dtype=BF, device="cuda", requires_grad=True)
    w = torch.nn.Parameter(torch.empty(512, dtype=BF, device="cuda"))
    cos = torch.empty(8, 32, device="cuda")
    at = torch.empty(3, dtype=torch.int32, device="cuda")
    lora = LoRALinear(XotLinear(512, 64, bias=False, device="cuda", dtype=BF), rank=2)
    assert not train_ops.takes(x) and not train_ops.takes(x, w)
    assert not train_ops.takes_heads(x, cos, cos, at, 64)
    assert not lora._takes(x)


def test_fake_tensors_are_not_read_by_linears():
  from types import SimpleNamespace
  from xotorch_amd import ops
  from xotorch_amd.models.llama import MLP, MoEMLP, XotLinear
  cfg = SimpleNamespace(dim=64, n_experts=2, n_experts_per_tok=1, moe_intermediate_dim=64, intermediate_dim=64)
  with FakeTensorMode(), torch.no_grad(), torch.device("cuda"):
    torch.set_default_dtype(BF)
    lin, mlp, moe = XotLinear(64, 128), MLP(cfg), MoEMLP(cfg)
    torch.set_default_dtype(torch.float32)
    for rows in (1, 3, 200):
      x = torch.empty(rows, 64, dtype=BF)
      assert not ops.few_rows(x, lin.weight) and not ops.tile_rows(x, lin.weight)
      assert lin(x).shape == (rows, 128)
    assert moe._grouped(torch.empty(300, 64, dtype=BF)) is None and moe._grouped(torch.empty(3, 64, dtype=BF)) is None


def test_products_go_where_they_are_faster():
  """Weights too wide for one round of blocks are the library's for many rows."""
  from xotorch_amd import ops
  for N, K in ((12288, 12288), (14336, 12288), (18432, 16384), (16384, 53248)):
    assert ops.parts_win(16, N, K) and ops.parts_win(17, N, K) == ops.parts_win(64, N, K) == (K != 16384)
    assert not ops.parts_win(65, N, K) and not ops.parts_win(256, N, K)
    assert not any(ops.tile_wins(m, N, K) for m in (17, 64, 65, 256))
  for N, K in ((4608, 3584), (8192, 28672), (10240, 8192), (3072, 2048)):
    assert all(ops.parts_win(m, N, K) for m in (1, 16, 17, 128, 129, 256))
  assert ops.tile_wins(128, 4096, 4096) and not ops.tile_wins(128, 2048, 2048) and ops.tile_wins(64, 2048, 2048)
  assert ops.tile_wins(256, 4096, 14336) and not ops.tile_wins(129, 3072, 2048)
  assert ops.tile_wins(64, 28672, 4096) and not ops.tile_wins(65, 28672, 4096) and not ops.tile_wins(17, 17920, 1536)
  assert not ops.tile_wins(4, 8192, 8192) and ops.tile_wins(128, 8192, 8192)
  assert ops.copy_pays(57344, 8192) and ops.copy_pays(12288, 28672) and not ops.copy_pays(8192, 28672) and not ops.copy_pays(28672, 4096)
  assert ops.gate_wins(128, 57344, 8192) and not ops.gate_wins(129, 57344, 8192)
  assert ops.gate_wins(64, 17920, 1536) and not ops.gate_wins(65, 17920, 1536) and ops.gate_wins(128, 16384, 2048)


@pytest.mark.parametrize("model_id", ["llama-3-8b", "gemma2-9b", "deepseek-v2-lite"])
def test_packing_without_a_gpu(model_id):
  from xotorch_amd.models import model_class_for
  from xotorch_amd.models.config import config_from_hf
  from xotorch_amd.models.registry import builtin_config
  from xotorch_amd.shard import Shard
  cfg = config_from_hf(builtin_config(model_id), model_id)
  with torch.device("meta"):
    model = model_class_for(cfg)(cfg, Shard(model_id, 1, 1, cfg.n_layers))
  assert model.pack_decode_weights() == 0


@pytest.mark.gpu
def test_only_copies_that_are_read():
  """One layer of the sizes of a 70B decoder: a copy of what tiles always do is not made,
  one that was made is among what is timed for steps of 64 rows."""
  from xotorch_amd import ops
  from xotorch_amd.engine.kvcache import make_cache
  from xotorch_amd.models import llama
  from xotorch_amd.models.config import config_from_hf
  from xotorch_amd.models.registry import builtin_config
  from xotorch_amd.shard import Shard
  cfg = config_from_hf(builtin_config("llama-3-70b"), "llama-3-70b")
  shard = Shard("llama-3-70b", 3, 3, cfg.n_layers)
  with torch.device("meta"):
    model = llama.ShardedModel(cfg, shard)
  model = model.to(BF).to_empty(device="cuda").eval()
  model.reset_rope()
  g = torch.Generator(device="cuda").manual_seed(0)
  with torch.inference_mode():
    for p in model.parameters():
      p.normal_(0, 0.02, generator=g) if p.dim() > 1 else p.fill_(1)
    model.pack_decode_weights()
    mlp, attn = model.layers["3"].mlp, model.layers["3"].self_attn
    assert mlp.gate_up_proj.weight_packed is not None
    assert all(m.weight_packed is None for m in (mlp.down_proj, attn.qkv_proj, attn.o_proj))
    x = torch.randn(64, 1, cfg.dim, generator=g, device="cuda").to(BF)
    found = []
    for copies in (True, False):
      cache = make_cache(cfg, shard, 64, 32, BF, "cuda")
      at = torch.zeros(1, dtype=torch.int32, device="cuda")
      if not copies:
        mlp.gate_up_proj.unpack_decode()
      found.append(model(x, caches=cache.caches, positions=at, start_pos=-1, is_decode=True,
                         seq_lens=torch.ones(64, dtype=torch.int32, device="cuda")).float())
    assert ("gate", 57344, 8192, 64) in llama._PACKED_WINS
    assert (found[0] - found[1]).norm() <= 0.01 * found[1].norm()
    y = mlp.gate_up_proj(x)
    mlp.gate_up_proj.pack_decode()
    assert (mlp.gate_up_proj(x).float() - y.float()).norm() <= 0.01 * y.float().norm()
    assert (57344, 8192, 64) in llama._PACKED_WINS


@pytest.mark.gpu
def test_the_rules_know_how_k_is_split():
  from xotorch_amd import ops
  for N in (1, 64, 65, 896, 1536, 4608, 8192, 9536, 9537, 14336, 14337, 28672, 28673, 151936, 1 << 26):
    for K in (64, 192, 256, 960, 1024, 2048, 3584, 4032, 4096, 16384, 53248):
      assert ops.tile_splits(N, K) == ops._tile().tile_splits(N, K)


@pytest.mark.gpu
def test_small_weights_are_split_for_one_round():
  """Parts that the kernels make, beside those that the rules count: fewer of up to 20 10^6 numbers, where
  that fills a round of the chip, and one only where the rules say so."""
  from xotorch_amd import ops
  hip = ops._tile()
  for N, K, parts in [(3584, 3584, 4), (4608, 3584, 3), (6400, 1024, 2), (6336, 1024, 4), (8192, 2432, 2), (8192, 2496, 4),
                      (904, 4864, 16), (2044, 1536, 6), (66, 1024, 4), (28672, 4096, 1), (64, 128, 1)]:
    assert hip.parts_of(N, K) == parts
    if N % 4 == 0:
      x, w = torch.zeros(3, K, device="cuda", dtype=torch.bfloat16), torch.zeros(N, K, device="cuda", dtype=torch.bfloat16)
      assert ops.tile_parts(x, w).shape == (parts, 3, N)
  for N in (1, 64, 65, 896, 1536, 4608, 6336, 8192, 9536, 14336, 14337, 28672, 28673, 151936, 1 << 26):
    for K in (64, 192, 256, 448, 512, 960, 1024, 2048, 3584, 4032, 4096, 16384, 53248):
      assert hip.parts_of(N, K) <= ops.tile_splits(N, K) and (hip.parts_of(N, K) == 1) == (ops.tile_splits(N, K) == 1)


@pytest.mark.gpu
def test_the_rules_know_how_k_of_gates_is_split():
  from xotorch_amd import ops
  for N in (16, 1024, 10176, 10192, 16384, 16400, 20416, 20480, 20496, 28672, 1 << 26):
    for K in (64, 1024, 1088, 2048, 2112, 6144, 6208, 53248):
      assert ops.gate_splits(N, K) == ops._tile().gate_splits(N, K)


def test_rules_and_kernels_split_alike():
  """What Python's rules write out of the kernels', over all that these tell apart: parts of two blocks a CU, blocks that
  begin at different places of k, a round of small weights."""
  hip = pytest.importorskip("xotorch_amd.ops._hip_tile")
  from xotorch_amd import ops
  rng = random.Random(5)
  sizes = {(N, K) for N in (2112, 3584, 4090, 4096, 4608, 8192, 11008, 16384, 28672, 53248)
           for K in (2048, 4096, 5696, 6144, 8192, 9600, 11008, 12288, 14336, 16384, 18432, 18944, 28672, 28736, 53248)}
  sizes |= {(round(2 ** rng.uniform(0, 18)), 64 * round(2 ** rng.uniform(0, 10))) for _ in range(20000)}
  for N, K in sizes:
    assert ops.tile_splits(N, K) == hip.tile_splits(N, K), (N, K)
    assert ops.gate_splits(N, K) == hip.gate_splits(N, K), (N, K)
  assert len({hip.gate_splits(N, K) for N, K in sizes}) >= 12


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [136, 200, 256])
def test_the_rules_know_which_gated_tiles_make_a_round(rows):
  from xotorch_amd import ops
  edges = [f * t + d for t in (64, 128, 160, 256, 320) for f in (143, 199, 256) for d in (-8, 0, 8)]
  for N in (1792, 4864, 16384, 17920, 28672, 37888, 57344, 106496, *edges):
    one_round = ops.tile_splits(N, 4096) == 1 and ops._tile().gate_tile(N, rows) > 0
    assert ops.gate_wins(rows, N, 4096) == one_round


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 5])
def test_a_linear_that_is_followed(rows, monkeypatch):
  from torch.fx.experimental.proxy_tensor import make_fx
  from xotorch_amd import ops
  from xotorch_amd.models.llama import XotLinear
  lin = XotLinear(64, 128).cuda().to(BF)
  x, y = (torch.randn(rows, 64, device="cuda").to(BF) for _ in "xy")
  plain, ad = torch.nn.functional.linear, torch.autograd.forward_ad
  with torch.no_grad():
    ref = plain(y, lin.weight, lin.bias).float()
    close = {"atol": 0.02, "rtol": 2.0 ** -6}
    assert ops.tile_rows(x, lin.weight)
    assert torch.allclose(make_fx(lin)(x)(y).float(), ref, **close)
    assert torch.allclose(torch.jit.trace(lin, (x,))(y).float(), ref, **close)
    assert torch.allclose(torch.func.vmap(lin)(y[:, None])[:, 0].float(), ref, **close)
    with ad.dual_level():
      assert ad.unpack_dual(lin(ad.make_dual(x, y))).tangent is not None
    with torch.autocast("cuda", torch.float16):
      assert lin(x).dtype == torch.float16
    with monkeypatch.context() as m:
      m.setattr(torch._C, "_cuda_getDevice", lambda: 1)
      found = ops.few_rows(x, lin.weight), ops.tile_rows(x, lin.weight)
    assert found == (False, False)


@pytest.mark.gpu
def test_training_on_another_device_than_the_current_one(monkeypatch):
  """Launches go to the current device's stream: other tensors are torch's."""
  from xotorch_amd.ops import torch_ref, train_ops
  x = torch.randn(2, 16, 512, device="cuda").to(BF).requires_grad_(True)
  w = torch.ones(512, device="cuda", dtype=BF)
  cos, sin = torch_ref.rope_cos_sin(64, 16, 10000.0, device="cuda")
  at = torch.arange(16, dtype=torch.int32, device="cuda")
  assert train_ops.takes(x, w) and train_ops.takes_heads(x, cos, sin, at, 64)
  with monkeypatch.context() as m:
    m.setattr(torch._C, "_cuda_getDevice", lambda: 1)
    found = train_ops.takes(x, w), train_ops.takes_heads(x, cos, sin, at, 64)
  assert found == (False, False)


@pytest.mark.gpu
def test_a_training_pass_that_is_followed():
  """A tracer records what torch's operators do; a kernel would be a constant to it."""
  from torch.fx.experimental.proxy_tensor import make_fx
  from xotorch_amd import ops
  x, w = torch.randn(4, 64, device="cuda").to(BF).requires_grad_(True), torch.ones(64, device="cuda", dtype=BF)

  def f(t):
    return ops.rmsnorm(t, w, 1e-5)

  graph, other = make_fx(f)(x), torch.randn(4, 64, device="cuda").to(BF).requires_grad_(True)
  assert (graph(other).float() - f(other).float()).abs().max() < 0.05


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1,), (3, 1, 64), (2, 1, 1, 64), ()])
def test_norms_with_weights_of_another_shape(shape):
  """What torch broadcasts: a kernel would read D numbers from the first on."""
  from xotorch_amd import ops
  from xotorch_amd.ops import torch_ref
  x, r = (torch.randn(2, 3, 1, 64, device="cuda").to(BF).requires_grad_(True) for _ in "xr")
  w = torch.randn(shape, device="cuda").to(BF)
  assert torch.equal(ops.rmsnorm(x, w, 1e-5), torch_ref.rmsnorm(x, w, 1e-5))
  for a, b in zip(ops.rmsnorm_residual(x, r, w, 1e-5), torch_ref.rmsnorm_residual(x, r, w, 1e-5)):
    assert torch.equal(a, b)


def test_what_a_prompt_loads_is_built_for_it():
  """A first run in a fresh checkout compiles what linears of prompts run on."""
  from xotorch_amd.engine.trace import DECODER
  from xotorch_amd.models.llama import XotLinear
  from xotorch_amd.ops.build import EXTENSIONS
  for needed in (DECODER, XotLinear.hip):
    assert {"_hip_rows", "_hip_tile", "_hip_gemm"} <= set(needed) <= set(EXTENSIONS)


def test_gradients_of_inputs_go_where_they_are_faster():
  """Many tokens only by long sums or small weights; a second tile of rows not by the largest."""
  from xotorch_amd.ops.train_ops import input_wins
  for N, K in ((2048, 2048), (4096, 14336), (16384, 2048), (28672, 4096), (128256, 2048)):
    assert all(input_wins(m, N, K) for m in (1, 40, 256, 300)) and (N < K or all(input_wins(m, N, K) for m in (666, 1000, 1001, 1400)))
  assert input_wins(1024, 8192, 8192) and not input_wins(1025, 8192, 8192)
  for N, K in ((4096, 4096), (6144, 4096), (5120, 3072)):
    assert input_wins(1280, N, K) and not input_wins(1281, N, K) and not input_wins(1401, N, K)
  assert input_wins(256, 8192, 28672) and not input_wins(257, 8192, 28672) and not input_wins(301, 4096, 14336)
  assert input_wins(2800, 16384, 2048) and not input_wins(2801, 16384, 2048) and input_wins(3000, 37888, 3584) and not input_wins(3001, 37888, 3584)


def test_products_that_later_tiles_gained():
  """Long sums, small weights of many tokens and ordinary weights of up to 2000; gradients of inputs of up to 8192."""
  from xotorch_amd.ops.train_ops import forward_gains, input_gains
  for M, N, K, own in [(64, 8192, 8064, False), (65, 8192, 8064, True), (1000, 8192, 8064, True), (1001, 8192, 8064, False),
                       (2000, 6144, 8064, True), (2001, 6144, 8064, False),
                       (1100, 8192, 28672, True), (1101, 8192, 28672, False), (1541, 8192, 28672, True), (1793, 8192, 28672, False),
                       # as blocks of 256 rows by 224 tokens fill rounds, whatever the width
                       (1344, 8192, 28672, False), (1345, 8192, 28672, True), (1792, 8192, 28672, True), (1600, 6400, 20480, False), (1793, 6400, 20480, True),
                       (1344, 9216, 24576, False), (1345, 9216, 24576, True), (1569, 9216, 24576, False), (1568, 7168, 18432, False), (1569, 7168, 18432, True),
                       (1300, 12288, 28672, True), (2000, 16384, 53248, True), (2001, 16384, 53248, False), (1001, 12288, 16384, False),
                       (8192, 5120, 17408, True), (8193, 5120, 17408, False),
                       (8192, 8192, 28672, False), (1000, 2048, 3072, False), (1001, 2048, 3072, True), (8192, 2048, 3072, True), (128, 28672, 4096, False),
                       (129, 28672, 4096, True), (2000, 28672, 4096, True), (2001, 28672, 4096, False), (100, 6144, 4096, True), (100, 16384, 2048, False),
                       (1500, 892, 2048, False), (1500, 2048, 832, False), (1500, 2050, 2048, False), (1500, 2048, 2056, False), (1500, 128256, 2048, False)]:
    assert forward_gains(M, N, K) == own, (M, N, K)
  for M, N, K, own in [(8192, 28672, 4096, True), (8193, 28672, 4096, False), (1, 896, 57344, True), (1, 896, 57352, False), (1, 832, 4096, False),
                       (1, 960, 900, False), (1, 928, 904, False), (4096, 128256, 4096, False)]:
    assert input_gains(M, N, K) == own, (M, N, K)


@pytest.mark.parametrize("needs", [(True, False), (False, True), (True, True)])
def test_a_linear_holds_what_its_gradients_read(needs):
  """Rows for the weight's gradient, the weight for that of the rows, as torch's operator; what is
  not held may change between the passes."""
  from xotorch_amd.ops import train_ops
  x, w, dy = (torch.randn(*s).to(BF) for s in ((2, 3, 40), (24, 40), (2, 3, 24)))
  x, w = x.requires_grad_(needs[0]), w.requires_grad_(needs[1])
  held, leaves = [], [t for t in (x, w) if t.requires_grad]
  with torch.autograd.graph.saved_tensors_hooks(lambda t: held.append(t.shape) or t, lambda t: t):
    y = train_ops.linear(x, w)
  assert sorted(held) == sorted(t.shape for t, other in ((x, w), (w, x)) if other.requires_grad)
  want = [(dy.flatten(0, 1) @ w.detach()).view_as(x), dy.flatten(0, 1).t() @ x.detach().flatten(0, 1)]
  first = torch.autograd.grad(y, leaves, dy.requires_grad_(), create_graph=True)
  assert all(torch.equal(a, b) for a, b in zip(first, [g for g, n in zip(want, needs) if n]))
  assert torch.autograd.grad(first[0].float().sum(), dy)[0].shape == dy.shape
  y = train_ops.linear(x, w)
  with torch.no_grad():
    for t, other in ((x, w), (w, x)):
      if not other.requires_grad:
        t.zero_()
  for a, b in zip(torch.autograd.grad(y, leaves, dy.detach()), first):
    assert torch.equal(a, b)


def test_products_of_more_rows_than_kernels_index():
  from xotorch_amd.ops import train_ops
  most = 1 << 22
  assert train_ops.forward_wins(64, 64, most) and train_ops.input_wins(64, most, 64) and train_ops.weight_wins(most, 64, 64)
  for more in (most + 8, most + 64):
    assert not train_ops.forward_wins(300, 4, more) and not train_ops.input_wins(64, more, 64) and not train_ops.weight_wins(more, 64, 64)


def test_products_of_a_vocabulary():
  from xotorch_amd.ops import train_ops
  for M, N, K, own in [(64, 128256, 2048, False), (65, 128256, 2048, True), (1000, 128256, 4096, True), (1001, 128256, 4096, False),
                       (300, 128256, 4160, False), (300, 100_000, 896, True), (300, 99_996, 896, False), (300, 151_938, 896, False)]:
    assert train_ops.forward_wins(M, N, K) == own, (M, N, K)
