// Products of training passes and prompts (bf16, fp32 sums) of some hundred to some thousand tokens:
//   forward           y = x W^T     [M, N] = [M, K] [N, K]^T
//   input_gradient    dx = dy W     [M, K] = [M, N] [N, K]
//   weight_gradient   dW = dy^T x   [N, K] = [M, N]^T [M, K]
// (The reference trains through torch's own operators, train/trainer of its engines.)
//
// What bounds them is the matrix cores, and how many blocks there are for them: library
// tiles leave most of the chip idle where results are small and sums long. Tiles are
// walked by mfma_tile.h; an operand whose rows lie along the sum is read as columns, by
// transposing reads from LDS, so that nothing is transposed in memory. Where tiles are few
// the sum is cut into parts, whose fp32 sums a second kernel adds up.
//
// us, library beside, weights from memory, 666 tokens: input [16384 -> 2048] 53 (117),
// [128256 -> 2048] 318 (869); weights [16384, 2048] 51 (63), [2048, 2048] 11 (20), [3584, 3584]
// 23 (32); forward [8192 -> 2048] 41 (43). 4096 tokens: weights [28672, 4096] 731 (812); input
// and forward of it 666 (675) and 670 (599).
#include "mfma_tile.h"

struct GemmArgs {
  const bf16_t *w, *x;  // y[m][n] = sum over k of x(m, k) w(n, k)
  void* y;              // bf16 [M, N], or fp32 [splits, M, N]
  int M, N, K;
  int steps, splits, group;  // steps of 64; tiles of x that are neighbours in a run of blocks
  const float *low, *by;     // y += scale low [M, rp] by [rank, N], or none
  int rank, rp;
  float scale;
};

// Where a wave's loads of an operand come from: rows [free, k] or, COL, columns [k, free]
template <bool COL, int F, int COUNT>
struct Source {
  static constexpr int SLOTS = F / 8, ROWS = COL ? 64 / SLOTS : 8;  // of a load: pieces of 16 bytes of a row, rows
  const char* base;     // of the tile, or of the wave's first load of columns, at the sum's first step
  size_t row;           // bytes from a k to the next
  unsigned next;        // and from a load of columns to the next
  unsigned off[COUNT];  // this lane's bytes besides
  DEVINL Source(const bf16_t* p, int f0, int free, int K, int wave, int lane) {
    const int load = wave * COUNT;
    if (COL) {
      base = (const char*)(p + (size_t)(load * ROWS) * free);
      row = (size_t)free * 2;
      next = ROWS * free * 2;
#pragma unroll
      for (int i = 0; i < COUNT; ++i) {
        const int slot = lane % SLOTS, f = f0 + (slot ^ col_turn((load + i) * ROWS + lane / SLOTS) << 1) * 8;
        off[i] = (lane / SLOTS * free + min(f, free - 8)) * 2;
      }
    } else {
      base = (const char*)(p + (size_t)f0 * K);
      row = 2;
      next = 0;
#pragma unroll
      for (int i = 0; i < COUNT; ++i) {
        const int r = (load + i) * 8 + (lane >> 3);
        off[i] = ((unsigned)min(r, free - 1 - f0) * K + ((lane & 7) ^ (r & 7)) * 8) * 2;
      }
    }
  }
  // the step that begins at k, if one is left: all of columns' rows may lie more than 4 GB apart
  DEVINL StepSource step(int k, int left) const {
    return COL ? StepSource(base + (k & StepSource::there(left)) * row, 0, left) : StepSource(base, k * 2, left);
  }
  // number I of it
  template <int I>
  DEVINL void load(StepSource from, char* to) const {
    if (COL) from.at = I * next & from.mask;
    from.load(off[I], to);
  }
};

template <bool COL, int N, int F> struct Operand { typedef RowFrags<N> Frags; };
template <int N, int F> struct Operand<true, N, F> { typedef ColFrags<N, F> Frags; };

// A block has BN of N and BM of M; WN waves along N. Eight waves, as blocks are few and short (mfma_tile.h), but
// four where the rows of x do not go by eight into pieces of 16 or the tile has too few of them
constexpr int waves_of(int bn, int bm) { return bm % 64 || bn * bm < 128 * 128 ? 4 : 8; }

// The low-rank term of an adapted linear, by fp32 products of the matrix cores (16 x 16 x 4), where a block's
// sums are whole: results go to memory once, and a pass that adds to them there reads and writes all of them
// again. us of 4096 tokens, rank 8, library and pass, this kernel and pass, so: [4096 -> 28672] 732, 763, 694, its
// input's gradient 711, 699, 686; [14336 -> 4096] 322, 336, 319, its input's gradient 435, 427, 394. Operands
// of eight features at once were 0 to 3% slower.
template <int R, int C>
DEVINL void add_low(floatx4 (&acc)[R][C], const GemmArgs& a, int m0, int n0, int lane) {
  const int col = lane & 15, quad = lane >> 4;
  for (int r0 = 0; r0 < a.rp; r0 += 4) {
    const int r = r0 + quad;
    const float* by = a.by + (size_t)min(r, a.rank - 1) * a.N;
    float w[R], x[C];
#pragma unroll
    for (int i = 0; i < R; ++i) w[i] = by[min(n0 + i * 16 + col, a.N - 1)];
#pragma unroll
    for (int j = 0; j < C; ++j) x[j] = a.low[(size_t)min(m0 + j * 16 + col, a.M - 1) * a.rp + r];
#pragma unroll
    for (int i = 0; i < R; ++i) w[i] = r < a.rank ? w[i] * a.scale : 0.f;
#pragma unroll
    for (int j = 0; j < C; ++j)
#pragma unroll
      for (int i = 0; i < R; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[j], acc[i][j], 0, 0, 0);
  }
}

template <bool WCOL, bool XCOL, int BN, int BM, int WN, int WB, int XB, bool PARTS, int WAVES = waves_of(BN, BM)>
__global__ __launch_bounds__(WAVES * 64) void gemm_kernel(GemmArgs a) {
  typedef MfmaTile<BN, BM, WN, WB, XB, WAVES> Sh;
  constexpr int R = Sh::R, C = Sh::C, WL = Sh::WL, XL = Sh::XL;
  extern __shared__ __attribute__((aligned(256))) bf16_t buf[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // blocks go round the eight dies: a die has a run of them, in panels of `group` tiles of
  // x that read the same of w
  const int nts = (a.N + BN - 1) / BN, mts = (a.M + BM - 1) / BM, die = blockIdx.x & 7, at = blockIdx.x >> 3;
  const int units = nts * mts * a.splits, rest = units & 7;
  if (at >= (units >> 3) + (die < rest)) return;
  const int unit = die * (units >> 3) + min(die, rest) + at, split = unit / (nts * mts), in_split = unit % (nts * mts);
  const int panel = in_split / (a.group * nts), in = in_split % (a.group * nts), wide = min(a.group, mts - panel * a.group);
  const int m0 = (panel * a.group + in % wide) * BM, n0 = in / wide * BN;
  const int s0 = (int)((long long)a.steps * split / a.splits), s1 = (int)((long long)a.steps * (split + 1) / a.splits);
  const Source<WCOL, BN, WL> ws(a.w, n0, a.N, a.K, wave, lane);
  const Source<XCOL, BM, XL> xs(a.x, m0, a.M, a.K, wave, lane);
  // the last step of columns ends where they do: what the one before has too is left out
  const int skip = WCOL && XCOL && s1 == a.steps ? a.steps * 64 - a.K : 0;
  auto k_of = [&](int s) { return WCOL && XCOL ? min((s0 + s) * 64, a.K - 64) : (s0 + s) * 64; };
  auto stepw = [&](int s) { return ws.step(k_of(s), s1 - s0 - s); };
  auto stepx = [&](int s) { return xs.step(k_of(s), s1 - s0 - s); };
  auto loadw = [&](auto number, const StepSource& from, unsigned to) {
    constexpr int i = decltype(number)::value;
    ws.template load<i>(from, (char*)buf + to + (wave * WL + i) * 1024);
  };
  auto loadx = [&](auto number, const StepSource& from, unsigned to) {
    constexpr int i = decltype(number)::value;
    xs.template load<i>(from, (char*)buf + to + (wave * XL + i) * 1024);
  };
  floatx4 acc[R][C];
  const int wr = wave % WN * (R * 16), wx = wave / WN * (C * 16);
  const unsigned base = (unsigned)(size_t)(lds_void*)buf;
  walk<Sh>(acc, typename Operand<WCOL, R, BN>::Frags(base, wr, lane), typename Operand<XCOL, C, BM>::Frags(base + Sh::XAT, wx, lane),
           s1 - s0, stepw, loadw, stepx, loadx, skip);
  if constexpr (!XCOL)
    if (a.low && split == 0) add_low(acc, a, m0 + wx, n0 + wr, lane);
  typedef typename std::conditional<PARTS, float, bf16_t>::type Out;
  const RowsOut<Out, R * 16> rows(buf, wave, lane);
#pragma unroll
  for (int j = 0; j < C; ++j) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int f = i * 16 + (lane >> 4) * 4;
      if constexpr (PARTS) rows.put(lane & 15, f, acc[i][j]);
      else rows.put(lane & 15, f, ushort4_t{f2b(acc[i][j][0]), f2b(acc[i][j][1]), f2b(acc[i][j][2]), f2b(acc[i][j][3])});
    }
    rows.out([&](int r, int f, floatx4 v) {
      const int m = m0 + wx + j * 16 + r, n = n0 + wr + f;
      if (m < a.M) st_piece((Out*)a.y + ((size_t)split * a.M + m) * a.N + n, v, a.N - n, a.N);
    });
  }
}

// bf16 of the parts' sums, in order; n % 4 == 0
__global__ __launch_bounds__(256) void parts_kernel(const float* __restrict__ part, bf16_t* __restrict__ y, size_t n, int splits) {
  for (size_t at = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4; at < n; at += (size_t)gridDim.x * 1024) {
    const floatx4 s = sum_parts(part, at, n, splits);
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = s[r];
    st4(y + at, v);
  }
}

// ===========================================================================
// host side
// ===========================================================================
template <bool WCOL, bool XCOL, int BN, int BM, int WN, int WB, int XB>
static void launch_gemm(const GemmArgs& a) {
  const int units = (a.N + BN - 1) / BN * ((a.M + BM - 1) / BM) * a.splits;
  constexpr int WAVES = waves_of(BN, BM), lds = MfmaTile<BN, BM, WN, WB, XB, WAVES>::LDS;
  auto run = [&](auto kernel) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    TORCH_CHECK(e == hipSuccess, "no LDS for a product's tiles");
    hipLaunchKernelGGL(kernel, dim3((units + 7) / 8 * 8), dim3(WAVES * 64), lds, cur_stream(), a);
  };
  if (a.splits > 1) run(gemm_kernel<WCOL, XCOL, BN, BM, WN, WB, XB, true>);
  else run(gemm_kernel<WCOL, XCOL, BN, BM, WN, WB, XB, false>);
}

// Tile and parts by what a round of the chip's 256 CUs takes, us: so much for a step of 64
// and for a block's begin and end, and the parts' sums once out and in again.
struct Tile {
  int bn, bm;
  double step, ends;
};
struct Costs {
  const Tile* tiles;
  int count;
  double bytes_us, parts;
};
// Of x as rows, fitted to 243 products of 64 to 4096 rows: a tile and parts within 1.3% of the fastest
// of these on average, 16% at most. With 256 and 128 rows of x alone it were 5%, and 13% of a tile's work
// is for rows that are not there at 666 tokens, whose products take, us, before and now: [2048 -> 128256] 370
// and 325, its gradient 360 and 315, [8192 -> 2048] 38.2 and 33.0. Small tiles are for weights that have
// few: blocks for all CUs without parts of the sum. [2048 -> 2048] 150, 333 and 1000 tokens 14.8 and 10.7, 15.3 and
// 11.2, 17.7 and 12.8, its gradient 15.0 and 11.4, 16.4 and 13.8, 19.0 and 15.0. Tiles of 160 rows of x, of 224 by
// 128 and of 64 by 64 gave less than 1% more. The last is for weights as rows alone: columns have no such form.
static const Tile ROW_TILES[] = {{256, 256, 1.14, 4.4}, {128, 256, 0.66, 2}, {256, 128, 0.76, 2}, {128, 128, 0.47, 1.3}, {256, 224, 0.95, 5.9},
                                 {256, 192, 0.93, 3.1}, {128, 192, 0.59, 2.9}, {128, 96, 0.44, 1.3}, {128, 64, 0.32, 1.2}, {64, 128, 0.26, 1.3}};
// As columns, of the first four tiles: within 8% of the fastest.
static const Tile COLUMN_TILES[] = {{256, 256, 1.42, 11}, {128, 256, 0.8, 7.5}, {256, 128, 0.8, 7.5}, {128, 128, 0.45, 4.7}};
struct Choice {
  int tile, splits;
};
// At every call, and passes of few tokens wait for the host: what all tiles share is made once, and nothing
// divides where they are compared: 0.32 us of [2048, 8192], 0.77 with divisions.
static Choice choose(const Costs& of, int64_t M, int64_t N, int steps) {
  double sum[16], way[16];  // by parts: steps of one, and the parts' way out and in
  int most = 0;
  for (int s = 1; s <= 16 && (s == 1 || (steps >= 4 * s && M * N * s <= 1 << 27)); ++s, ++most) {
    sum[most] = (unsigned)(steps + s - 1) / (unsigned)s;
    way[most] = s > 1 ? M * N * 8.0 * s / of.bytes_us + of.parts : 0;
  }
  Choice best{0, 1};
  double least = 1e30;
  for (int t = 0; t < of.count; ++t) {
    const Tile& tile = of.tiles[t];
    const int64_t blocks = (int64_t)((unsigned)(N + tile.bn - 1) / (unsigned)tile.bn) * ((unsigned)(M + tile.bm - 1) / (unsigned)tile.bm);
    for (int i = 0; i < most; ++i) {
      const double us = (double)((blocks * (i + 1) + 255) >> 8) * (sum[i] * tile.step + tile.ends) + way[i];
      if (us < least) least = us, best = {t, i + 1};
    }
  }
  return best;
}

// y [M, N] of x [M, K] (XCOL: [K, M]) and w [N, K] (WCOL: [K, N]), and scale low by if they are given
template <bool WCOL, bool XCOL>
static Tensor product(const Tensor& x, const Tensor& w, const OptT& low = {}, const OptT& by = {}, double scale = 1) {
  check_io(x, torch::kBFloat16);
  check_io(w, torch::kBFloat16);
  CHK(x.dim() == 2 && w.dim() == 2);
  const int64_t m = x.size(XCOL), N = w.size(WCOL), K = x.size(!XCOL);
  CHK(K == w.size(!WCOL) && m >= 1 && N >= 1 && K >= 1 && m <= 1 << 22 && N <= 1 << 22 && K <= 1 << 22);
  CHK(((size_t)x.data_ptr() & 15) == 0 && ((size_t)w.data_ptr() & 15) == 0);
  // whole pieces of 16 bytes, and steps of the sum: columns' last may begin in the one before
  CHK(XCOL ? K >= 64 && m % 8 == 0 : K % 64 == 0);
  CHK(WCOL ? N % 8 == 0 : N % 4 == 0);
  GemmArgs a{};
  a.x = P<bf16_t>(x);
  a.w = P<bf16_t>(w);
  a.M = (int)m;
  a.N = (int)N;
  a.K = (int)K;
  a.steps = (int)((K + 63) / 64);
  if (low) {
    CHK(by.has_value() && !XCOL);
    check_io(*low, torch::kFloat32);
    check_io(*by, torch::kFloat32);
    CHK(low->dim() == 2 && by->dim() == 2 && low->size(0) == m && by->size(1) == N && by->size(0) >= 1 && by->size(0) <= 16);
    a.rank = (int)by->size(0);
    a.rp = a.rank <= 4 ? 4 : a.rank <= 8 ? 8 : 16;
    CHK(low->size(1) == a.rp);
    a.low = P<float>(*low);
    a.by = P<float>(*by);
    a.scale = (float)scale;
  }
  // us of [4096, 28672 x 4096], panels of 2, 4 and 8 tiles of x: 694, 675, 676; 8192 of all, 766, 733, 723
  a.group = 4;
  const Costs of = XCOL ? Costs{COLUMN_TILES, 4, 5e6, 2.5} : Costs{ROW_TILES, WCOL ? 9 : 10, 7.2e6, 4};
  const Choice c = choose(of, m, N, a.steps);
  a.splits = c.splits;
  CHK((N / of.tiles[c.tile].bn + 1) * (m / of.tiles[c.tile].bm + 1) * a.splits <= INT_MAX / 8);
  auto y = torch::empty({m, N}, x.options());
  Tensor part;
  a.y = y.data_ptr();
  if (a.splits > 1) {
    part = f32(x, {a.splits, m, N});
    a.y = part.data_ptr();
  }
  if (c.tile == 0) launch_gemm<WCOL, XCOL, 256, 256, 2, 3, 2>(a);
  else if (c.tile == 1) launch_gemm<WCOL, XCOL, 128, 256, 2, 3, 3>(a);
  else if (c.tile == 2) launch_gemm<WCOL, XCOL, 256, 128, 4, 3, 3>(a);
  else if (c.tile == 3) launch_gemm<WCOL, XCOL, 128, 128, 2, 4, 4>(a);
  else if constexpr (!XCOL) {
    if (c.tile == 4) launch_gemm<WCOL, XCOL, 256, 224, 2, 3, 2>(a);
    else if (c.tile == 5) launch_gemm<WCOL, XCOL, 256, 192, 2, 3, 2>(a);
    else if (c.tile == 6) launch_gemm<WCOL, XCOL, 128, 192, 2, 4, 4>(a);
    else if (c.tile == 7) launch_gemm<WCOL, XCOL, 128, 96, 2, 4, 4>(a);
    else if (c.tile == 8) launch_gemm<WCOL, XCOL, 128, 64, 2, 4, 4>(a);
    else if constexpr (!WCOL) launch_gemm<WCOL, XCOL, 64, 128, 1, 4, 4>(a);
  }
  if (a.splits > 1) {
    const size_t n = (size_t)m * N;
    hipLaunchKernelGGL(parts_kernel, dim3(std::min<size_t>((n + 1023) / 1024, 4096)), dim3(256), 0, cur_stream(), part.data_ptr<float>(),
                       M<bf16_t>(y), n, a.splits);
  }
  return y;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("forward", [](Tensor x, Tensor w, OptT low, OptT by, double scale) { return product<false, false>(x, w, low, by, scale); },
        "x w^T of x [M, K], w [N, K], and scale low by of narrow rows and [rank, N]", py::arg("x"), py::arg("w"), py::arg("low") = py::none(),
        py::arg("by") = py::none(), py::arg("scale") = 1.0);
  m.def("input_gradient", [](Tensor dy, Tensor w, OptT low, OptT by, double scale) { return product<true, false>(dy, w, low, by, scale); },
        "dy w of dy [M, N], w [N, K], and scale low by of narrow rows and [rank, K]", py::arg("dy"), py::arg("w"), py::arg("low") = py::none(),
        py::arg("by") = py::none(), py::arg("scale") = 1.0);
  m.def("weight_gradient", [](Tensor dy, Tensor x) { return product<true, true>(dy, x); }, "dy^T x of dy [M, N], x [M, K]");
}
