"""Products of a few rows (hip/rows_ops.hip) against 64 bits, at the edges of row
groups (4 weight rows), of steps along k (512) and of the row counts that it takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (rows, N, K): less than a group, remainders of both, rows split over the waves of a block or not
SIZES = [(1, 1, 8), (2, 3, 40), (2, 5, 512), (1, 130, 520), (1, 8196, 1536), (2, 16386, 1544), (1, 8200, 2048),
         (2, 9, 4104), (1, 66, 18944)]


def _inputs(m, N, K, seed=0):
  g = torch.Generator(device="cuda").manual_seed(seed)
  x, w, n, r = (torch.randn(*s, generator=g, device="cuda") for s in ((m, K), (N, K), (K,), (m, N)))
  return x, w.to(torch.bfloat16), (1 + 0.1 * n).to(torch.bfloat16), r


def _check(y, ref, terms, K, rounded):
  """terms: sum of the products' sizes. Sums of K products in fp32 are off by less than K 2^-24 of
  it; `rounded`: operands that are rounded to bf16 by half of 2^-8 (a third of a step left for the norm's own)."""
  bound = terms * (K * 2.0 ** -24 + (2.0 ** -8 if rounded else 0)) + ref.abs() * (2.0 ** -8 if y.dtype == torch.bfloat16 else 2.0 ** -22)
  assert y.shape == ref.shape and bool(((y.double() - ref).abs() <= bound + 1e-30).all())


@pytest.mark.parametrize("m,N,K", SIZES)
def test_products(m, N, K):
  from xotorch_amd import ops
  x, w, _, r = _inputs(m, N, K)
  x, bias = x.to(torch.bfloat16), r[0].to(torch.bfloat16)
  ref, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
  with torch.no_grad():
    assert ops.few_rows(x, w)
    _check(ops.rows_linear(x, w), ref, terms, K, False)
    _check(ops.rows_linear(x, w, bias), ref + bias.double(), terms + bias.double().abs(), K, False)
    rb = r.to(torch.bfloat16)
    for res, dt in ((r, torch.bfloat16), (rb, torch.float32)):
      y = ops.rows_add_linear(x, w, res)
      assert y.dtype == dt
      # the product as bf16: half of 2^-8 of it; an fp32 residual likewise
      more = ref.abs() * 2.0 ** -8 + (res.double().abs() * 2.0 ** -8 if res is r else 0)
      assert bool(((y.double() - ref - res.double()).abs()
                   <= more + terms * K * 2.0 ** -24 + (ref + res.double()).abs() * 2.0 ** (-8 if res is r else -22)).all())


@pytest.mark.parametrize("m,N,K", SIZES[:-1] + [(2, 12, 32768)])
def test_products_of_normed_rows(m, N, K):
  from xotorch_amd import ops
  x, w, n, _ = _inputs(m, 2 * N, K, seed=1)
  xb = x.to(torch.bfloat16)
  with torch.no_grad():
    assert ops.few_rows_normed(xb, (n,), w)
    for add in (0.0, 1.0):
      def normed(v):
        v = v.double()
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-5) * (n.double() + add)
      h = normed(xb)
      _check(ops.rows_norm_linear(xb, n, 1e-5, w, None, add), h @ w.double().t(), h.abs() @ w.double().abs().t(), K, True)
      h = normed(x)
      (g, u), (tg, tu) = (h @ w.double().t()).chunk(2, -1), (h.abs() @ w.double().abs().t()).chunk(2, -1)
      act = torch.nn.functional.silu
      # |d silu| <= 1.1 |d g|
      err = 1.1 * tg * (K * 2.0 ** -24 + 2.0 ** -8)
      bound = err * (u.abs() + tu * 2.0 ** -7) + act(g).abs() * tu * (K * 2.0 ** -24 + 2.0 ** -8) + (act(g) * u).abs() * 2.0 ** -8
      bound += (1.1 * g.abs() * u.abs() + act(g).abs() * u.abs()) * 2.0 ** -8  # gate and up as bf16
      assert bool(((ops.rows_norm_swiglu(x, n, 1e-5, w, add).double() - act(g) * u).abs() <= bound + 1e-30).all())


def test_infinite_weights_stay_in_their_row():
  """What lies past a row's end is not multiplied with anything."""
  from xotorch_amd import ops
  w = torch.ones(9, 520, device="cuda", dtype=torch.bfloat16)
  w[3, -1], w[5, 0] = float("inf"), float("nan")
  x = torch.ones(2, 520, device="cuda", dtype=torch.bfloat16)
  with torch.no_grad():
    y = ops.rows_linear(x, w)
  want = torch.full((2, 9), 520.0, device="cuda", dtype=torch.bfloat16)
  want[:, 3], want[:, 5] = float("inf"), float("nan")
  assert torch.equal(y.nan_to_num(nan=-1.0), want.nan_to_num(nan=-1.0))


def test_other_rows_go_the_general_way():
  from xotorch_amd import ops
  w = torch.ones(8, 16, device="cuda", dtype=torch.bfloat16)
  x = torch.ones(2, 16, device="cuda", dtype=torch.bfloat16)
  assert not ops.few_rows(x, w)  # under grad
  with torch.no_grad():
    assert ops.few_rows(x, w)
    assert not ops.few_rows(torch.ones(3, 16, device="cuda", dtype=torch.bfloat16), w)
    assert not ops.few_rows(x.float(), w) and not ops.few_rows(x.t(), w) and not ops.few_rows(x[:, :12].contiguous(), w[:, :12])
    assert not ops.few_rows(torch.ones(33, device="cuda", dtype=torch.bfloat16)[1:].view(2, 16), w)
    assert not ops.few_rows(x[:0], w) and not ops.few_rows(x, w[:, 1:9])


def test_one_row_summed_as_more_are():
  from xotorch_amd import ops
  from xotorch_amd.models.llama import XotLinear
  lin = XotLinear(4096, 512, bias=False).cuda().to(torch.bfloat16)
  x = torch.randn(5, 4096, generator=torch.Generator(device="cuda").manual_seed(0), device="cuda").to(torch.bfloat16)
  with torch.inference_mode():
    assert ops.few_rows(x[:1], lin.weight)
    with ops.sums_of_more_rows():
      assert not ops.few_rows(x[:1], lin.weight)
      assert torch.equal(lin(x)[:1], lin(x[:1]))
    assert ops.few_rows(x[:1], lin.weight)


# blocks with several row groups, whose waves have none, one, two, three or nine steps of each, and rows about
# as long as what a thread keeps of them (2048 and 4096 numbers)
@pytest.mark.parametrize("m,N,K", [(1, 9000, 264), (1, 20000, 600), (2, 9000, 1032), (1, 8300, 2056), (2, 8300, 2048), (1, 4200, 4096),
                                   (2, 8300, 4104)])
def test_further_row_groups(m, N, K):
  test_products_of_normed_rows(m, N, K)
