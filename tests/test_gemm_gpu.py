"""Products of training passes and prompts (hip/gemm_ops.hip) against 64 bits: rows and features at the
edges of tiles, sums of one step, of whole ones and of what is left, cut into parts or not."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# tokens, features out and in: tiles of 128 and 256 and a few past them, few tiles (parts) and many
SIZES = [(64, 64, 64), (65, 72, 128), (127, 520, 64), (200, 128, 1032), (257, 384, 256), (666, 3072, 2048),
         (333, 16384, 264), (100, 8192, 136), (1001, 256, 4096), (1400, 1536, 896), (70, 40960, 1024), (640, 24, 8)]


def _random(seed, *shape):
  g = torch.Generator(device="cuda").manual_seed(seed)
  return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)


def _near(got, a, b):
  """got is a b^T: fp32 sums of K products, less than K 2^-24 of their sizes off, stored as bf16."""
  want, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
  assert got.shape == want.shape
  return bool(((got.double() - want).abs() <= size * (a.shape[1] + 8) * 2.0 ** -24 + want.abs() * 2.0 ** -8 + 1e-30).all())


@pytest.mark.parametrize("M,N,K", SIZES)
def test_products(M, N, K):
  from xotorch_amd.ops import train_ops
  hip = train_ops._hip_gemm()
  x, w, dy = _random(M, M, K), _random(N, N, K), _random(K, M, N)
  if K % 64 == 0 and N % 4 == 0:
    assert _near(hip.forward(x, w), x, w)
  if N % 64 == 0:
    assert _near(hip.input_gradient(dy, w), dy, w.t())
  assert _near(hip.weight_gradient(dy, x), dy.t(), x.t())


# rows of 4 numbers more than pieces of 8: whole sums and parts of them, tiles of 128 and 256
@pytest.mark.parametrize("M,N,K", [(65, 68, 128), (300, 4100, 192), (100, 260, 4096), (1001, 12, 64), (700, 18308, 128), (2048, 516, 2048),
                                   (65, 128256, 128), (300, 100_004, 64), (1000, 151936, 64)])  # the last three a vocabulary's
def test_products_of_half_pieces(M, N, K):
  from xotorch_amd.ops import train_ops
  x, w = _random(M, M, K), _random(N, N, K)
  assert _near(train_ops._hip_gemm().forward(x, w), x, w)


@pytest.mark.parametrize("M,N,K", [(191, 16392, 2048), (385, 8200, 4096), (192, 4104, 8192),  # 128 x 192, then in parts
                                   (385, 33000, 128), (450, 16388, 128), (129, 8200, 8192),  # 256 x 192
                                   (221, 33000, 1024), (448, 24584, 1024), (666, 2048, 65536),  # 256 x 224
                                   (95, 16392, 320), (577, 4100, 64), (129, 2048, 8192),  # 128 x 96
                                   (65, 1032, 64), (385, 4104, 128), (192, 4104, 4096),  # 128 x 64
                                   (570, 2052, 320), (127, 8200, 4096), (1, 68, 8192), (193, 1032, 4096)])  # 64 x 128 (and gradients by 128 x 64)
def test_tiles_between(M, N, K):
  """Tiles of other shapes than 128 and 256: one row short, full, a tile for a few, sums in parts."""
  from xotorch_amd.ops import train_ops
  hip = train_ops._hip_gemm()
  x, w = _random(M, M, K), _random(N, N, K)
  assert _near(hip.forward(x, w), x, w)
  if N % 8 == 0:
    assert _near(hip.input_gradient(x, w.t().contiguous()), x, w)


@pytest.mark.parametrize("M,N,K,rank", [(1, 72, 64, 1), (65, 1032, 64, 4), (570, 2056, 320, 5), (193, 1032, 4096, 8), (385, 4104, 128, 9),
                                        (95, 16392, 320, 16), (129, 2048, 8192, 8), (385, 8200, 4096, 16), (450, 16392, 128, 3), (129, 8200, 8192, 8),
                                        (221, 33000, 1024, 8), (666, 2048, 65536, 16), (1300, 4104, 320, 8), (383, 16392, 320, 2),
                                        (2100, 4096, 4096, 8), (95, 8200, 8192, 8), (383, 8200, 64, 8)])
def test_low_rank_terms(M, N, K, rank):
  """Of adapters, added inside the products, of every tile, in parts or not; numbers past the rank and the ends count
  for nothing. Not rounded before the sum: fp32 products of K + rank numbers."""
  from xotorch_amd.ops import train_ops
  hip = train_ops._hip_gemm()
  x, w = _random(M, M, K), _random(N, N, K)
  g = torch.Generator(device="cuda").manual_seed(rank)
  by = torch.randn(rank, N, generator=g, device="cuda")
  low = torch.zeros(M, 4 if rank <= 4 else 8 if rank <= 8 else 16, device="cuda")
  low[:, :rank] = torch.randn(M, rank, generator=g, device="cuda") * K ** 0.5
  want = x.double() @ w.double().t() + 0.75 * low[:, :rank].double() @ by.double()
  size = x.double().abs() @ w.double().abs().t() + 0.75 * low[:, :rank].double().abs() @ by.double().abs()
  for got in (hip.forward(x, w, low, by, 0.75), hip.input_gradient(x, w.t().contiguous(), low, by, 0.75)):
    assert bool(((got.double() - want).abs() <= size * (K + rank + 9) * 2.0 ** -24 + want.abs() * 2.0 ** -8).all())


@pytest.mark.parametrize("left", [64, 65, 127, 128, 129, 1003])
def test_what_is_left_of_a_sum_counts_once(left):
  """Tokens past whole steps; infinities in rows that the last step has twice stay what they are."""
  from xotorch_amd.ops import train_ops
  x, dy = _random(1, left, 136), _random(2, left, 264)
  assert _near(train_ops._hip_gemm().weight_gradient(dy, x), dy.t(), x.t())
  x[left - 60, 3] = float("inf")
  dy[left - 60] = 1.0
  got = train_ops._hip_gemm().weight_gradient(dy, x)
  want = dy.float().t() @ x.float()
  assert torch.equal(got.isfinite(), want.isfinite()) and torch.equal(got.isinf(), want.isinf())


@pytest.mark.parametrize("form", ["rows", "batch", "one", "turned", "shifted", "weight shifted", "weight turned", "spread"])
def test_linears_of_all_forms(form):
  """Gradients of a linear whatever the strides and alignments of what it is given."""
  from xotorch_amd import ops
  from xotorch_amd.ops import train_ops
  M, N, K = (70, 128, 192) if form != "one" else (1, 128, 192)
  x, w, dy = _random(1, M, K), _random(2, N, K), _random(3, M, N)
  if form == "batch":
    x, dy = x.view(7, 10, K), dy.view(7, 10, N)
  if form == "one":
    x, dy = x[0], dy[0]
  if form == "turned":
    x = x.t().contiguous().t()
  if form == "shifted":
    x = torch.cat([x.new_zeros(1), x.flatten()])[1:].view(M, K)
  if form == "weight shifted":
    w = torch.cat([w.new_zeros(1), w.flatten()])[1:].view(N, K)
  if form == "weight turned":
    w = w.t().contiguous().t()
  if form == "spread":
    dy = dy[:, :1].expand(M, N)
  x, w = x.detach().requires_grad_(), w.detach().requires_grad_()
  assert train_ops.takes_linear(x, w)
  held = []
  with torch.autograd.graph.saved_tensors_hooks(lambda t: held.append(t.shape) or t, lambda t: t):
    y = ops.linear(x, w)
  assert len(held) == 2 and y.shape == dy.shape
  dx, dw = torch.autograd.grad(y, (x, w), dy)
  rows, drows = x.detach().reshape(-1, K), dy.reshape(-1, N)
  assert dx.shape == x.shape and dw.shape == w.shape
  assert _near(y.detach().reshape(-1, N), rows, w.detach()) and _near(dx.reshape(-1, K), drows, w.detach().t()) and _near(dw, drows.t(), rows.t())


def test_linears_that_others_follow():
  """Second derivatives, functorch and forward mode are torch's operators'."""
  from torch.func import vmap
  from xotorch_amd import ops
  x, w = _random(1, 70, 64).requires_grad_(), _random(2, 128, 64).requires_grad_()
  dx, = torch.autograd.grad(ops.linear(x, w).float().square().sum(), x, create_graph=True)
  (again,) = torch.autograd.grad(dx.float().sum(), w)
  assert again.isfinite().all()
  assert vmap(lambda t: ops.linear(t, w))(x[None]).shape == (1, 70, 128)
  with torch.autograd.forward_ad.dual_level():
    y = ops.linear(torch.autograd.forward_ad.make_dual(x.detach().float(), torch.ones_like(x).float()), w.detach().float())
    assert torch.autograd.forward_ad.unpack_dual(y).tangent is not None


@pytest.mark.parametrize("rank", [0, 8, 20])
def test_backward_passes_that_others_follow(rank):
  """A dispatch mode around the backward pass alone sees its products."""
  from torch.utils._python_dispatch import TorchDispatchMode
  from xotorch_amd import ops
  from xotorch_amd.models.llama import XotLinear
  from xotorch_amd.train.lora import LoRALinear
  seen = []

  class Recorder(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
      seen.append(func.overloadpacket)
      return func(*args, **(kwargs or {}))

  x, w, dy = _random(1, 300, 256).requires_grad_(), _random(2, 512, 256), _random(3, 300, 512)
  if rank:
    lin = LoRALinear(XotLinear(256, 512, bias=False).to("cuda", torch.bfloat16), rank=rank)
    lin.base.weight.data.copy_(w)
    y, leaves = lin(x), (x, lin.lora_a, lin.lora_b)
  else:
    w.requires_grad_()
    y, leaves = ops.linear(x, w), (x, w)
  with Recorder():
    found = torch.autograd.grad(y, leaves, dy)
  products = [f for f in seen if f in (torch.ops.aten.mm, torch.ops.aten.addmm, torch.ops.aten.addmm_)]
  assert len(products) >= (4 if rank else 2)
  assert _near(found[0], dy, w.detach().t())  # B is zero
  if not rank:
    assert _near(found[1], dy.t(), x.detach().t())


@pytest.mark.parametrize("M", [70, 300])
def test_many_gradients_at_once(M):
  from xotorch_amd import ops
  from xotorch_amd.ops import train_ops
  x, w, dy = _random(1, M, 192).requires_grad_(), _random(2, 128, 192).requires_grad_(), _random(3, 2, M, 128)
  assert train_ops.takes_linear(x, w)
  dx, dw = torch.autograd.grad(ops.linear(x, w), (x, w), dy, is_grads_batched=True)
  for i in range(2):
    assert _near(dx[i], dy[i], w.detach().t()) and _near(dw[i], dy[i].t(), x.detach().t())


@pytest.mark.parametrize("M,N,K,form", [(257, 64, 64, "rows"), (300, 4096, 192, "batch"), (1000, 520, 2048, "turned"),
                                        (512, 2048, 8192, "shifted"), (260, 72, 128, "weight shifted"), (333, 128, 64, "weight turned"),
                                        (512, 8192, 12352, "rows"), (2000, 128, 16448, "rows"), (1000, 6144, 12352, "rows")])
def test_linears_of_prompts(M, N, K, form):
  from xotorch_amd import ops
  from xotorch_amd.ops import train_ops
  x, w = _random(1, M, K), _random(2, N, K)
  if form == "batch":
    x = x.view(M // 10, 10, K)
  if form == "turned":
    x = x.t().contiguous().t()
  if form == "shifted":
    x = torch.cat([x.new_zeros(1), x.flatten()])[1:].view(M, K)
  if form == "weight shifted":
    w = torch.cat([w.new_zeros(1), w.flatten()])[1:].view(N, K)
  if form == "weight turned":
    w = w.t().contiguous().t()
  with torch.inference_mode():
    assert train_ops.takes_product(x, w) and not train_ops.takes_product(x.reshape(-1, K)[:256], w)
    y = ops.linear(x, w)
    with torch.autocast("cuda", torch.float16):
      assert not train_ops.takes_product(x, w)
  assert y.shape == (*x.shape[:-1], N) and _near(y.reshape(-1, N), x.reshape(-1, K), w)


@pytest.mark.parametrize("M,N,K,form", [(65, 4100, 8064, "rows"), (2000, 4160, 8064, "turned"), (8192, 896, 16448, "rows"), (1001, 896, 896, "batch"),
                                        (8192, 1920, 960, "spread"), (129, 4160, 2560, "shifted"), (2000, 9028, 896, "weight shifted"),
                                        (300, 9024, 1024, "weight turned"), (70, 8192, 3264, "rows"), (1500, 960, 904, "batch"), (1100, 896, 57344, "rows")])
def test_linears_that_later_tiles_gained(M, N, K, form):
  """At the ends of train_ops.forward_gains and input_gains, whatever the strides and alignments."""
  from xotorch_amd import ops
  from xotorch_amd.ops import train_ops
  assert train_ops.forward_gains(M, N, K) > train_ops.forward_wins(M, N, K) or train_ops.input_gains(M, N, K) > train_ops.input_wins(M, N, K)
  x, w, dy = _random(1, M, K), _random(2, N, K), _random(3, M, N)
  if form == "batch":
    x, dy = x[None], dy[None]
  if form == "turned":
    x = x.t().contiguous().t()
  if form == "shifted":
    x = torch.cat([x.new_zeros(1), x.flatten()])[1:].view(M, K)
  if form == "weight shifted":
    w = torch.cat([w.new_zeros(1), w.flatten()])[1:].view(N, K)
  if form == "weight turned":
    w = w.t().contiguous().t()
  if form == "spread":
    dy = dy[:, :1].expand(M, N)
  x = x.detach().requires_grad_()
  y = ops.linear(x, w)
  dx, = torch.autograd.grad(y, x, dy)
  assert y.shape == dy.shape and dx.shape == x.shape
  rows, drows = x.detach().reshape(-1, K), dy.reshape(-1, N)
  assert _near(y.detach().reshape(-1, N), rows, w) and _near(dx.reshape(-1, K), drows, w.t())
  if M > 256:
    with torch.inference_mode():
      assert _near(ops.linear(x, w).reshape(-1, N), rows, w)


@pytest.mark.parametrize("M,N,K,form", [(257, 32, 64, "rows"), (320, 288, 128, "batch"), (513, 4096, 192, "shifted"), (1000, 2080, 448, "turned"),
                                        (2305, 1536, 64, "rows"), (769, 9728, 896, "rows"), (300, 512, 8192, "rows")])
def test_gates_of_prompts(M, N, K, form):
  """silu(x gate^T) (x up^T) against 64 bits: even shares of rows, tiles cut in two, features past a tile's."""
  from xotorch_amd.ops import train_ops
  x, w = _random(1, M, K), _random(2, N, K)
  if form == "batch":
    x = x.view(M // 10, 10, K)
  if form == "turned":
    x = x.t().contiguous().t()
  if form == "shifted":
    x = torch.cat([x.new_zeros(1), x.flatten()])[1:].view(M, K)
  with torch.inference_mode():
    assert train_ops.takes_gate(x, w) and not train_ops.takes_gate(x.reshape(-1, K)[:256], w) and not train_ops.takes_gate(x, w[:, :K - 8])
    y = train_ops.gate_product(x, w)
  assert y.shape == (*x.shape[:-1], N // 2)
  rows = x.reshape(-1, K).double()
  (gate, up), (by_gate, by_up) = (rows @ w.double().t()).chunk(2, 1), (rows.abs() @ w.double().abs().t() * (K + 8) * 2.0 ** -24).chunk(2, 1)
  silu = gate * torch.sigmoid(gate)  # its slope is less than 1.1
  bound = 1.1 * by_gate * (up.abs() + by_up) + silu.abs() * by_up + (silu * up).abs() * 2.0 ** -8
  assert bool(((y.reshape(-1, N // 2).double() - silu * up).abs() <= bound + 1e-30).all())


# more and fewer rows a tile than rows / 256 makes, whole and cut in two
@pytest.mark.parametrize("M,N", [(257, 9728), (300, 17920), (513, 16384), (600, 16384), (700, 16384), (1000, 17920), (1200, 16416)])
def test_gates_of_prompts_in_even_rounds(M, N):
  test_gates_of_prompts(M, N, 128, "rows")


def test_gates_of_prompts_in_a_layer():
  """One kernel where nobody waits for the product, with the module's hooks and its graph."""
  from xotorch_amd.models.llama import MLP
  from xotorch_amd.models.registry import builtin_config
  from xotorch_amd.models import config_from_hf
  m = MLP(config_from_hf(builtin_config("llama-3.2-1b"), "m"), 1024).to("cuda", torch.bfloat16)
  x, seen = _random(3, 300, m.gate_up_proj.in_features), []
  with torch.no_grad():
    assert m.whole_gate(x) and not m.whole_gate(x[:256])
    y = m(x)
    hook = m.gate_up_proj.register_forward_hook(lambda *a: seen.append(1))
    want = m(x)
    hook.remove()
    assert seen == [1]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
      again = m(x)
    for _ in range(3):
      again.zero_()
      g.replay()
      assert torch.equal(again, y)
  assert ((y - want).float().norm() / want.float().norm()).item() < 2.0 ** -7  # bf16 gate and up, then twice as many roundings
  x.requires_grad_()
  assert not m.whole_gate(x)
  m(x).float().sum().backward()
  assert x.grad is not None
