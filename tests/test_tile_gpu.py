"""Products by weight tiles (hip/tile_ops.hip) against 64 bits: rows at the edges of
16, 32, 64 and 128, weight rows past a tile, k with and without a split."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(1, 8, 64), (16, 72, 320), (17, 130, 1536), (32, 2048, 2048), (33, 136, 512), (64, 3584, 3584), (65, 129, 128),
         (128, 520, 18944), (129, 2056, 640), (256, 28680, 192), (129, 28680, 64), (200, 3592, 3584)]


def _inputs(m, N, K):
  g = torch.Generator(device="cuda").manual_seed(m)
  return [torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16) for s in ((m, K), (N, K), (N,))]


@pytest.mark.parametrize("m,N,K", SIZES)
def test_products(m, N, K):
  """Sums of K products in fp32 are off by less than K 2^-24 of the products' sizes;
  what is stored as bf16 by 2^-8 of itself."""
  from xotorch_amd import ops
  x, w, b = _inputs(m, N, K)
  ref, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t() * (K * 2.0 ** -24)
  with torch.no_grad():
    assert ops.tile_rows(x, w)
    parts = ops.tile_parts(x, w)
    assert parts.shape[1:] == ref.shape and bool(((parts.double().sum(0) - ref).abs() <= terms).all())
    for bias in (None, b):
      want = ref if bias is None else ref + b.double()
      y = ops.tile_linear(x, w, bias)
      assert bool(((y.double() - want).abs() <= terms + want.abs() * 2.0 ** -8 + 1e-30).all())
    if N % 8 == 0:
      (g, u), (tg, tu) = ref.chunk(2, -1), (terms + ref.abs() * 2.0 ** -8).chunk(2, -1)
      act = torch.nn.functional.silu(g)
      bound = 1.1 * tg * (u.abs() + tu) + act.abs() * tu + (act * u).abs() * 2.0 ** -8
      assert bool(((ops.tile_swiglu(x, w).double() - act * u).abs() <= bound + 1e-30).all())


# from 65 rows on: parts of few steps and of many, blocks for a round, for more than one and for
# half of one, rows of x in two blocks, weight rows past a tile and off the 16 bytes of a piece
@pytest.mark.parametrize("m,N,K", [(66, 3592, 3584), (100, 4104, 14336), (128, 1002, 8192), (128, 33000, 128), (81, 41000, 64), (150, 3084, 4096),
                                   (192, 4104, 1536), (193, 4100, 2048), (219, 28364, 128), (122, 47436, 192), (130, 1000, 1024), (256, 1006, 512), (160, 57352, 128), (129, 65528, 64)])
def test_products_of_more_rows(m, N, K):
  test_products(m, N, K)


# parts that make one round of blocks of 64 weight rows, for each number of rows of x
@pytest.mark.parametrize("m", [16, 65, 128, 129, 192, 193, 256])
@pytest.mark.parametrize("N,K", [(3584, 3584), (2044, 1536), (4600, 4288), (8192, 2432), (1024, 1088), (904, 4864), (66, 1024)])
def test_products_in_a_round_of_parts(m, N, K):
  test_products(m, N, K)


# one part more than 448 blocks take, where two a CU are all there; not where seven parts turn; nor of half as many tiles
@pytest.mark.parametrize("N,K,splits", [(3584, 5696, 9), (4090, 6208, 8), (4096, 14336, 7), (2048, 11008, 14)])
def test_two_blocks_a_cu(N, K, splits):
  from xotorch_amd.ops import _hip_tile
  assert _hip_tile.parts_of(N, K) == splits
  for m in (3, 40, 130):
    test_products(m, N, K)


@pytest.mark.parametrize("N,K", [(72, 320), (3584, 3584), (28680, 192), (520, 18944), (1048, 4096), (264, 16384),
                                 (40968, 4096), (40960, 4096), (36872, 4096)])  # the last five begin at different places of k
def test_rows_do_not_depend_on_their_batch(N, K):
  from xotorch_amd import ops
  x, w, b = _inputs(256, N, K)
  with torch.no_grad():
    whole = ops.tile_linear(x, w, b), ops.tile_swiglu(x, w)
    for lo, hi in ((0, 1), (3, 19), (40, 72), (100, 164), (7, 135), (20, 200)):
      some = x[lo:hi].contiguous()
      assert torch.equal(ops.tile_linear(some, w, b), whole[0][lo:hi]) and torch.equal(ops.tile_swiglu(some, w), whole[1][lo:hi])


@pytest.mark.parametrize("m,D,parts", [(1, 8, 1), (3, 2048, 4), (5, 2056, 16), (256, 8192, 3), (2, 16384, 2)])
def test_sum_and_norm(m, D, parts):
  from xotorch_amd import ops
  g = torch.Generator(device="cuda").manual_seed(D)
  p = torch.randn(parts, m, D, generator=g, device="cuda")
  x, w = (torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16) for s in ((m, D), (D,)))
  total = p[0]
  for q in p[1:]:
    total = total + q
  f = x.float() + total.to(torch.bfloat16).float()
  for rounded in (False, True):
    h, n = ops.parts_add_norm(p, x, w, 1e-5, 1.0, rounded)
    assert torch.equal(h, f.to(torch.bfloat16))
    v = (h if rounded else f).double()
    ref = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-5) * (w.double() + 1)
    # bf16 once, and fp32 sums of D squares
    assert bool(((n.double() - ref).abs() <= ref.abs() * (2.0 ** -8 + D * 2.0 ** -24) + 1e-30).all())
  assert torch.equal(ops.parts_add_norm(p, x)[0], f.to(torch.bfloat16))


# weight rows that make one round of tiles of 128, 160 and 256; steps of k around the buffers' number
@pytest.mark.parametrize("m,N,K", [(65, 36872, 64), (128, 40968, 192), (104, 65536, 384), (136, 25480, 128), (193, 32768, 256),
                                   (136, 31856, 128), (256, 40960, 320), (193, 50952, 64), (256, 65528, 192)])
def test_gated_products_of_one_round(m, N, K):
  from xotorch_amd import ops
  x, w, _ = _inputs(m, N, K)
  w = w * K ** -0.5
  with torch.no_grad():
    assert ops.gate_wins(m, N, K)
    y = ops.tile_swiglu(x, w).double()
  ref, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t() * (K * 2.0 ** -24)
  (g, u), (tg, tu) = ref.chunk(2, -1), (terms + ref.abs() * 2.0 ** -8).chunk(2, -1)  # products are stored as bf16 would be
  act = torch.nn.functional.silu(g)
  bound = 1.1 * tg * (u.abs() + tu) + act.abs() * tu + (act * u).abs() * 2.0 ** -8
  assert bool(((y - act * u).abs() <= bound + 1e-30).all())


# 64 weight rows a block: a feature, a tile and a round of them less, just so and more; rows of
# x of one tile and of several; whole rows 2 KB and 4 KB apart
@pytest.mark.parametrize("N,K", [(16, 64), (72, 1024), (2056, 704), (10256, 2048), (16384, 2048), (16400, 128), (9728, 896)])
def test_gated_products_of_whole_rows(N, K):
  from xotorch_amd import ops
  assert ops._tile().gate_splits(N, K) == 1
  x, w, _ = _inputs(256, N, K)
  ref = x.double() @ w.double().t()
  size = x.double().abs() @ w.double().abs().t()
  with torch.no_grad():
    all_rows = ops.tile_swiglu(x, w)
    for m in (3, 17, 33, 64, 65, 100, 128, 129, 193):
      assert torch.equal(ops.tile_swiglu(x[:m].contiguous(), w), all_rows[:m])
  gate, up = ref.chunk(2, -1)
  # each product is rounded to 8 bits after fp32 sums of K; silu's slope is at most 1.1
  by = 2.0 ** -8
  dg, du = (p.abs() * by + s * (K + 8) * 2.0 ** -24 for p, s in zip(ref.chunk(2, -1), size.chunk(2, -1)))
  act = torch.nn.functional.silu(gate)
  slack = (1.1 * dg + gate.abs() * 2.0 ** -19) * (up.abs() + du) + act.abs() * du + (act * up).abs() * by
  assert bool(((all_rows.double() - act * up).abs() <= slack + 1e-30).all())


# weight rows that blocks of four to eight waves fill rounds best with, a tile's last ones missing
@pytest.mark.parametrize("N,waves", [(37872, 5), (17920, 5), (24560, 6), (22016, 6), (28656, 7), (49136, 4), (32752, 8), (49120, 4)])
def test_gated_products_fill_their_rounds(N, waves):
  from xotorch_amd import ops
  assert waves in {ops._tile().gate_waves(N, m) or (8 if m > 16 and N > 199 * 128 else 4) for m in (16, 32, 64)}
  for m in (1, 16, 17, 32, 33, 64):
    test_gated_product(m, N, 192)


def test_gated_product(m=5, N=25584, K=320):
  """Products rounded to bf16 after fp32 sums; silu's slope is at most 1.1."""
  from xotorch_amd import ops
  x, w, _ = _inputs(m, N, K)
  (g, u), (tg, tu) = (x.double() @ w.double().t()).chunk(2, -1), (x.double().abs() @ w.double().abs().t() * (K * 2.0 ** -24)).chunk(2, -1)
  tg, tu, act = tg + g.abs() * 2.0 ** -8, tu + u.abs() * 2.0 ** -8, torch.nn.functional.silu(g)
  bound = 1.1 * tg * (u.abs() + tu) + act.abs() * tu + (act * u).abs() * 2.0 ** -8
  with torch.no_grad():
    assert bool(((ops.tile_swiglu(x, w).double() - act * u).abs() <= bound + 1e-30).all())


@pytest.mark.parametrize("m,D,H,I", [(3, 64, 128, 192), (45, 2048, 2048, 8192), (200, 320, 192, 512)])
def test_rest_of_a_layer_is_its_parts(m, D, H, I):
  from xotorch_amd import ops
  g = torch.Generator(device="cuda").manual_seed(m)
  heads, x, post, after, wo, gu, down = (torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16) * s[-1] ** -0.5 for s in (
    (1, m, H), (1, m, D), (D,), (D,), (D, H), (2 * I, D), (D, I)))
  with torch.no_grad():
    h, n = ops.parts_add_norm(ops.tile_parts(heads, wo), x, post, 1e-5)
    want = ops.parts_add_norm(ops.tile_parts(ops.tile_swiglu(n, gu), down), h, after, 1e-6, rounded=True)
    got, alone = ops.tile_rest(heads, wo, x, post, 1e-5, gu, down, after, 1e-6), ops.tile_rest(heads, wo, x, post, 1e-5, gu, down)
  assert len(got) == 2 and len(alone) == 1 and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and torch.equal(alone[0], want[0])


# rows whose offsets take 32 bits just so, and more: by mfma_tile.h, and by several blocks of 64 rows of x each
@pytest.mark.parametrize("K", [1 << 22, (1 << 22) + 64])
@pytest.mark.parametrize("m,N", [(65, 8), (130, 8), (130, 6)])
def test_products_of_longest_rows(m, N, K):
  from xotorch_amd import ops
  g = torch.Generator(device="cuda").manual_seed(m + N)
  x = torch.randn(m, K, generator=g, device="cuda", dtype=torch.bfloat16)
  w = torch.randn(N, K, generator=g, device="cuda", dtype=torch.bfloat16) * 2.0 ** -11
  want = torch.stack([w.double() @ row.double() for row in x])
  # K / 32 additions of 32 products at most; sums of random signs stay within six standard deviations
  slack = x.norm(dim=1, keepdim=True, dtype=torch.float64) * w.norm(dim=1, dtype=torch.float64) * K ** -0.5 * 6 * (K / 32 + 8) * 2.0 ** -24
  with torch.no_grad():
    assert bool(((ops.tile_linear(x, w).double() - want).abs() <= slack + want.abs() * 2.0 ** -8).all())
    if N % 4 == 0:
      assert bool(((ops.tile_parts(x, w).double().sum(0) - want).abs() <= slack).all())
