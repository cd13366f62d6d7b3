// Products of up to 256 rows (decode batches, prompt chunks) with bf16 weights as
// they lie in the checkpoint, [N, K] row-major, and what follows them:
//   y = x W^T + bias; silu(x Wg^T) (x Wu^T); r + x W^T and the norm of it.
// (The reference runs these as separate modules, general_mha.py:83-102,
// llm_utils.py:465-500.)
//
// What bounds them is the weights' way from memory, for which every CU wants some
// 48 KB on its way; library tiles leave that to few blocks. A block owns 64 to 128
// weight rows and all rows of x (up to 64, more by mfma_tile.h), and walks its part of
// k in steps of 64 through a ring of LDS buffers that are filled by direct loads: rows of 128
// bytes, so whole lines, the 16-byte pieces of row r permuted by r & 7 in the global
// address, which spreads fragment reads over the banks. Where the weight rows alone
// make too few blocks, k is split; the parts' fp32 sums are added by the kernel that
// follows anyway (norm, activation).
//
// us, library beside: [3584, 18944] m 8 23 (46), m 32 23 (110), m 128 32 (99);
// [8192, 28672] m 128 88 (201); [8192, 8192] m 128 28 (47); [4608, 3584] m 256 16 (36).
//
// How k is split depends on the weights' shape alone, and the order of the sums within
// a part on the shape and the weight row: a row of these products does not depend on the
// rows beside it.
// (Whether a product is one of these does, and so does how attention cuts its keys.)
#include "common.h"
#include "stream_tile.h"

struct TileArgs {
  const bf16_t *x, *w, *bias;
  void* y;  // bf16 [m, N], or fp32 [splits, m, N]
  int m, N, K, splits;  // N: output features
  int turned;         // see first_step: 0, or how many features of a gated product begin together
  bool runs, dense;   // see run_tile, launch_tile
  int whole, more, inv;  // steps of 64 of a part, in all parts `more` besides; 65536 / splits, and one more
};

// All that a block needs to send its first loads, read at once: the compiler would leave
// half of it until it knows which tile this is, and wait for memory twice
DEVINL void read_args(const TileArgs& a) {
  asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.m), "s"(a.N), "s"(a.K), "s"(a.splits), "s"(a.whole), "s"(a.more), "s"(a.inv));
}

// A part's first step, steps * split / splits: up to 16 parts, no division
DEVINL int part_at(const TileArgs& a, int split) { return split * a.whole + (split * a.more * a.inv >> 16); }

// STORE: bf16 with bias; PART: fp32 sums of a part of k; GATED: weight rows [2 N, K],
// gate first, bf16 of the gated activation
enum TileEnd { STORE, PART, GATED };

// Where the blocks of weight rows (or GATED features) from `row` on begin among the `len`
// steps of their part of k. Blocks that walk k in step read the same columns of rows that
// lie a multiple of 8 KB apart, which few memory channels hold: where rows or parts do
// (turns), blocks begin at different places. It goes by weight rows, so that a row of x
// is summed up as in any other batch. us, all from the start of their part first:
// [8192, 8192] m 4 32, 22; m 128 35, 29; gate [57344, 8192] m 32 166, 145; [28672, 4096]
// m 4 42, 36; [4096, 14336] in 7 parts m 32 26, 19. Other lengths gain nothing
// ([37888, 3584] m 8 47.4, 47.9); long ones lose, whose parts of x come from L2 only while
// all blocks want the same ([8192, 28672] m 128 93, 115). Rows that begin together are
// whole tiles of any size that the weights may meet: where one is 160 rows (gate_tile), 640
// features.
template <int END>
DEVINL int first_step(const TileArgs& a, int row, int len) {
  if (!a.turned) return 0;
  const unsigned group = END != GATED ? (unsigned)row / 256 : a.turned == 640 ? (unsigned)row / 640 : (unsigned)row / 128;
  return (int)(((group * 2654435761u >> 16) * (unsigned)len) >> 16);
}

// A wave's sums of weight rows wr .. of a tile and rows m0 .. of x
template <int END, int BN, int R, int C>
DEVINL void finish_tile(const TileArgs& a, const floatx4 (&acc)[R][C], int tile, int split, int m0, int wr, int lane) {
  const int col = lane & 15, quad = lane >> 4;
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int m = m0 + j * 16 + col;
    if (END == GATED) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        // lanes of quads 0 and 1 hold gates, those of 2 and 3 the products of up
        const int n = tile * (BN / 2) + (wr + i * 16) / 2 + quad * 4;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = siluf(rounded(acc[i][j][r])) * rounded(__shfl_xor(acc[i][j][r], 32));
        if (m >= a.m || quad > 1) continue;
        bf16_t* dst = (bf16_t*)a.y + (size_t)m * a.N + n;
        if (n + 3 < a.N && (a.N & 3) == 0) st4(dst, v);
        else
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < a.N) st(dst + r, v[r]);
      }
    } else {
      if (m >= a.m) continue;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int n = tile * BN + wr + i * 16 + quad * 4;
        const bool whole = n + 3 < a.N && (a.N & 3) == 0;
        if (END == PART) {
          float* dst = (float*)a.y + ((size_t)split * a.m + m) * a.N + n;
          if (whole) *(floatx4*)dst = acc[i][j];
          else
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (n + r < a.N) dst[r] = acc[i][j][r];
        } else {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = acc[i][j][r] + (a.bias && n + r < a.N ? ld(a.bias + n + r) : 0.f);
          bf16_t* dst = (bf16_t*)a.y + (size_t)m * a.N + n;
          if (whole) st4(dst, v);
          else
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (n + r < a.N) st(dst + r, v[r]);
        }
      }
    }
  }
}

template <int BN, int BM, int BUFS, int END, int WAVES>
__global__ __launch_bounds__((TileShape<BN, BM, BUFS, WAVES>::WAVES * 64)) void tile_kernel(TileArgs a) {
  typedef TileShape<BN, BM, BUFS, WAVES> Sh;
  constexpr int R = Sh::R, C = Sh::C;
  extern __shared__ __attribute__((aligned(16))) bf16_t buf[];  // [BUFS][weights [BN][64], x [BM][64]]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  read_args(a);
  // blocks go round the eight dies: two blocks of the same weights are neighbours on one.
  // The grid says which part a block has, as divisions come before all loads: a product of 7
  // steps ([3584, 3584], 8 rows) took 7.6 us with three of them and takes 7.1
  const int mts = (a.m + BM - 1) / BM, tiles = (a.N + (END == GATED ? BN / 2 : BN) - 1) / (END == GATED ? BN / 2 : BN);
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int mt = mts > 1 ? local % mts : 0, at = mts > 1 ? local / mts : local;
  int split = blockIdx.y, tile = at * 8 + ((die - split * tiles) & 7);
  if (a.runs) {  // or a die has a run of them, and so few parts of x
    const int units = tiles * a.splits, rest = units & 7, n = at + split * ((tiles + 7) >> 3);
    if (n >= (units >> 3) + (die < rest)) return;
    split = (die * (units >> 3) + min(die, rest) + n) / tiles;
    tile = die * (units >> 3) + min(die, rest) + n - split * tiles;
  } else if (a.dense) {
    split = (at * 8 + die) / tiles;
    tile = at * 8 + die - split * tiles;
  }
  if (tile >= tiles || split >= a.splits) return;
  const int s0 = part_at(a, split), s1 = part_at(a, split + 1), m0 = mt * BM;
  const bf16_t *wsrc[Sh::WL], *xsrc[Sh::XL];
  const int sub = lane >> 3;
  // GATED: 8 gate rows and the same 8 up rows in turn
  auto weight_row = [&](int r) -> size_t {
    if (END == GATED) return (size_t)min(tile * (BN / 2) + (r >> 4) * 8 + (r & 7), a.N - 1) + ((r >> 3) & 1 ? (size_t)a.N : 0);
    return min(tile * BN + r, a.N - 1);
  };
#pragma unroll
  for (int i = 0; i < Sh::WL; ++i) {
    const int r = (wave * Sh::WL + i) * 8 + sub;
    wsrc[i] = a.w + weight_row(r) * a.K + ((lane & 7) ^ (r & 7)) * 8;
  }
#pragma unroll
  for (int i = 0; i < Sh::XL; ++i) {
    const int r = BM >= 32 ? ((wave & 3) * Sh::XL + i) * 8 + sub : (wave & 3) * 4 + (sub & 3);  // waves past four load the same again
    xsrc[i] = a.x + (size_t)min(m0 + r, a.m - 1) * a.K + ((lane & 7) ^ (r & 7)) * 8;
  }
  const int len = s1 - s0, turn = first_step<END>(a, tile * (END == GATED ? BN / 2 : BN), len);
  floatx4 acc[R][C];
  const int wr = Sh::wr(wave), wx = Sh::wx(wave);
#pragma unroll
  for (int i = 0; i < Sh::WL; ++i) wsrc[i] += s0 * 64;
#pragma unroll
  for (int i = 0; i < Sh::XL; ++i) xsrc[i] += s0 * 64;
  stream_walk<Sh>(acc, buf, wsrc, xsrc, len, turn, wave, lane);
  finish_tile<END, BN, R, C>(a, acc, tile, split, m0 + wx, wr, lane);
}

// The same of 65 to 256 rows of x, by mfma_tile.h. With 256 rows the weights' way from memory
// and that of x from L2 to every CU bound it: [37888, 3584] 46 us for the former alone, 61 for
// both without products, 65 with them.
template <int BN, int BM, int WN, int WB, int XB, int WAVES, int END>
__global__ __launch_bounds__((WAVES * 64)) void wide_kernel(TileArgs a) {
  typedef MfmaTile<BN, BM, WN, WB, XB, WAVES> Sh;
  constexpr int R = Sh::R, C = Sh::C, WL = Sh::WL, XL = Sh::XL, PER = END == GATED ? BN / 2 : BN;
  extern __shared__ __attribute__((aligned(16))) bf16_t buf[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int piece = ((lane & 7) ^ (lane >> 3)) * 8;
  read_args(a);
  // blocks go round the eight dies, or a die has a run of them (run_tile); those of the same
  // weights are neighbours
  const int tiles = (a.N + PER - 1) / PER, mts = a.m > BM ? (a.m + BM - 1) / BM : 1, units = tiles * a.splits * mts;
  const int die = blockIdx.x & 7, rest = units & 7;
  if ((int)(blockIdx.x >> 3) >= (units >> 3) + (die < rest)) return;
  const int n = a.runs ? die * (units >> 3) + min(die, rest) + (blockIdx.x >> 3) : blockIdx.x, unit = mts > 1 ? n / mts : n, m0 = (n - unit * mts) * BM;
  const int split = a.splits > 1 ? unit / tiles : 0, tile = unit - split * tiles, s0 = part_at(a, split), s1 = part_at(a, split + 1);
  // GATED: 8 gate rows and the same 8 up rows in turn, of which a wave loads either
  const int up = END == GATED ? wave / (WAVES / 2) : 0;
  const bf16_t *wsrc = a.w + ((size_t)tile * PER + (up ? (size_t)a.N : 0)) * a.K + s0 * 64, *xsrc = a.x + (size_t)m0 * a.K + s0 * 64;
  unsigned woff[WL], wto[WL], xoff[XL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int g = END == GATED ? wave % (WAVES / 2) * WL + i : wave * WL + i;
    woff[i] = ((unsigned)min(g * 8 + (lane >> 3), a.N - 1 - tile * PER) * a.K + piece) * 2;
    wto[i] = (END == GATED ? g * 2 + up : g) * 1024;
  }
#pragma unroll
  for (int i = 0; i < XL; ++i) xoff[i] = ((unsigned)min((wave * XL + i) * 8 + (lane >> 3), a.m - 1 - m0) * a.K + piece) * 2;
  const int len = s1 - s0, turn = first_step<END>(a, tile * PER, len);
  auto step = [&](const bf16_t* p, int s) { return StepSource(p, (s + turn < len ? s + turn : s + turn - len) * 128, len - s); };
  auto stepw = [&](int s) { return step(wsrc, s); };
  auto stepx = [&](int s) { return step(xsrc, s); };
  auto loadw = [&](auto number, const StepSource& from, unsigned at) {
    constexpr int i = decltype(number)::value;
    from.load<2>(woff[i], (char*)buf + at + wto[i]);
  };
  auto loadx = [&](auto number, const StepSource& from, unsigned at) {
    constexpr int i = decltype(number)::value;
    from.load(xoff[i], (char*)buf + at + (wave * XL + i) * 1024);
  };
  floatx4 acc[R][C];
  const int wr = wave % WN * (R * 16), wx = wave / WN * (C * 16), col = lane & 15, quad = lane >> 4;
  const unsigned base = (unsigned)(size_t)(lds_void*)buf;
  walk<Sh>(acc, RowFrags<R>(base, wr, lane), RowFrags<C>(base + Sh::XAT, wx, lane), len, stepw, loadw, stepx, loadx);
  typedef typename std::conditional<END == PART, float, bf16_t>::type Out;
  // GATED: two tiles of x at a time. Lanes of quads 0 and 1 hold gates, those of 2 and 3 the
  // products of up; changed round, lanes have both, the lower half those of the first tile.
  constexpr int N = END == GATED ? R * 8 : R * 16, PAIR = END == GATED ? 2 : 1;
  static_assert(C % PAIR == 0, "");
  const RowsOut<Out, N, PAIR * 16> rows(buf, wave, lane);
  const int n0 = tile * PER + (END == GATED ? wr / 2 : wr);
#pragma unroll
  for (int j = 0; j < C; j += PAIR) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if constexpr (END == GATED) {
        ushort4_t v;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i][j][r]), __float_as_uint(acc[i][j + 1][r]), false, false);
          v[r] = f2b(siluf(rounded(__uint_as_float(both[0]))) * rounded(__uint_as_float(both[1])));
        }
        rows.put((quad >> 1) * 16 + col, i * 8 + (quad & 1) * 4, v);
      } else if constexpr (END == PART) {
        rows.put(col, i * 16 + quad * 4, acc[i][j]);
      } else {
        const int n = n0 + i * 16 + quad * 4;
        ushort4_t v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = f2b(acc[i][j][r] + (a.bias && n + r < a.N ? ld(a.bias + n + r) : 0.f));
        rows.put(col, i * 16 + quad * 4, v);
      }
    }
    rows.out([&](int r, int f, floatx4 v) {
      const int m = m0 + wx + j * 16 + r;
      if (m < a.m) st_piece((Out*)a.y + ((size_t)split * a.m + m) * a.N + n0 + f, v, a.N - n0 - f, a.N);
    });
  }
}

// ---------------------------------------------------------------------------
// what follows a product whose k was split: the parts' sums, in order
// ---------------------------------------------------------------------------

// y = bf16 of the sums + bias; GATE: [m, 2 N] -> silu(gate) up [m, N]. N % 4 == 0.
template <bool GATE>
__global__ __launch_bounds__(256) void finish_kernel(const float* __restrict__ part, const bf16_t* __restrict__ bias,
                                                     bf16_t* __restrict__ y, int m, int N, int splits) {
  const int at = (blockIdx.x * 256 + threadIdx.x) * 4, wide = GATE ? 2 * N : N;
  if (at >= N) return;
  const size_t row = blockIdx.y, stride = (size_t)m * wide;
  const floatx4 g = sum_parts(part, row * wide + at, stride, splits);
  float v[4];
  if (GATE) {
    const floatx4 u = sum_parts(part, row * wide + N + at, stride, splits);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = siluf(rounded(g[r])) * rounded(u[r]);
  } else {
    float b[4] = {};
    if (bias) ld4(bias + at, b);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = g[r] + b[r];
  }
  st4(y + row * N + at, v);
}

// h = x + bf16 of the sums (bf16), n = norm(x + ..) w. One block a row, which stays
// in registers; with few rows its chain of loads is all the time there is, so that
// threads take 4 numbers (8 of rows over 4096). ROUND: the norm reads h as it is stored.
// 8 rows of 3584, 8 parts: 5 us (11 with 256 threads and part after part).
template <int NC, int THREADS>
__global__ __launch_bounds__(THREADS) void add_norm_kernel(const float* __restrict__ part, const bf16_t* __restrict__ x,
                                                       const bf16_t* __restrict__ w, bf16_t* __restrict__ h,
                                                       bf16_t* __restrict__ n, int m, int D, int splits, float eps,
                                                       float add, bool round) {
  __shared__ float red[THREADS / 64];
  const size_t row = (size_t)blockIdx.x * D, stride = (size_t)m * D;
  float v[NC][4], ss = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int at = (c * THREADS + threadIdx.x) * 4;
    if (at >= D) break;
    const floatx4 p = sum_parts(part, row + at, stride, splits);
    ld4(x + row + at, v[c]);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[c][r] += rounded(p[r]);
    st4(h + row + at, v[c]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (round) v[c][r] = rounded(v[c][r]);
      ss += v[c][r] * v[c][r];
    }
  }
  if (!w) return;
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int i = 0; i < THREADS / 64; ++i) ss += red[i];
  const float inv = rsqrtf(ss / (float)D + eps);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int at = (c * THREADS + threadIdx.x) * 4;
    if (at >= D) break;
    float by[4];
    ld4(w + at, by);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[c][r] *= inv * (by[r] + add);
    st4(n + row + at, v[c]);
  }
}

// ===========================================================================
// host side
// ===========================================================================
// Parts of tiles that don't go round the eight dies evenly are numbered through, at a division's
// cost: blocks without work between the others keep CUs from them, which then have two. us,
// parts of the grid and numbered through: [4608, 3584] in 36 tiles and 7 parts, m 20 10.7, 8.2;
// m 48 12.5, 9.3
template <int BN, int BM, int BUFS, int END, int WAVES = 4>
static void launch_tile(TileArgs a) {
  typedef TileShape<BN, BM, BUFS, WAVES> Sh;
  if (Sh::LDS > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)tile_kernel<BN, BM, BUFS, END, WAVES>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, Sh::LDS);
    TORCH_CHECK(e == hipSuccess, "no LDS for weight tiles");
  }
  const int per = END == GATED ? BN / 2 : BN;
  const int tiles = (a.N + per - 1) / per, mts = (a.m + BM - 1) / BM;
  a.dense = !a.runs && a.splits > 1 && tiles % 8;
  const dim3 grid = a.dense ? dim3((tiles * a.splits + 7) / 8 * 8 * mts) : dim3((tiles + 7) / 8 * 8 * mts, a.splits);
  hipLaunchKernelGGL((tile_kernel<BN, BM, BUFS, END, WAVES>), grid, dim3(Sh::WAVES * 64), Sh::LDS, cur_stream(), a);
}

// Tile and depth by the rows of x and by the blocks that 128 weight rows make. us at
// [N, K], 64-row or (deeper, fewer to a CU) first:
//   m 32: [2048, 2048] in 128 blocks 4.1, 4.6; [3584, 18944] in 224 25.0, 22.6
//   m 64: [2048, 2048] 4.6, 5.6; [28672 -> 8192] 91.0, 78.3
// From 65 rows of x on by mfma_tile.h, all rows in one block but where that leaves half of the
// chip idle. Up to 128: where blocks make one
// round and their sums are long, four waves and more on the way, else eight, two blocks to a
// CU; us, the former first (and by the loop above, m 128):
//   m 96 and 128: [8192, 28672] 79 and 87, 82 and 90 (89); gate [28672, 4096] 42 and 46, 51
//   and 50 (49); [3584, 3584] 10.2 and 11.0, 9.7 and 10.5 (11.2); [50304, 2048] in 393 blocks
//   m 128 58, 51 (53); gate [35840, 8192] in 280 blocks m 66 135, 129 (166)
// More rows in eight waves where they can be (from registers and with eight waves of the loop
// before: m 256 [3584, 3584] 15.7, now 14.4; [1536, 8960] 19.0, 14.9; [8192, 8192] 38.6,
// 37.1); with blocks for half of the chip and less, in two blocks of 128 ([2048, 2048] 8.8,
// in one 10.2).
//
// The gated product of more than 64 rows takes the weight tile that makes one round of the
// chip's 256 CUs, if there is one: [37888, 3584] 237 blocks of 160 rows 65 with m 256, 57
// with 136 (library and activation 84; waves of 80 by 128 68; 296 blocks of 128 120, 148 of
// 256 77); [57344, 8192] 224 of 256 196 with m 256 (220; 448 of 128 235), 165 with 192 in
// tiles that have no more (in those of 256 200). Up to 128 rows, whose matrix products are
// short, 148 blocks of 256 are enough: 63 with m 128 (73; 78).
static int gate_tile(int rows, int m) {
  if (m <= 128) return rows > 143 * 256 && rows <= 256 * 256 ? 256 : 0;
  for (int tile : {128, 160, 256})
    if (rows > 199 * tile && rows <= 256 * tile) return tile;
  return 0;
}

// Up to 64 rows: waves of a block, each of 16 weight rows, by how full the last of up to four rounds
// of 256 blocks is, where that is more than tiles of 64 or (8, also four waves) 128 rows fill it by
// 8%, or by 20% for more than 32 rows of x, which more waves read more often from LDS. us, by those
// first: [37888, 3584] m 8 48.7, 43.1, m 32 59.6, 46.0, m 64 66.1, 54.1; [17920, 1536] m 8 14.6, 12.5, m 45
// 19.1, 14.7; [49152, 3584] m 16 57.2, 57.3, m 24 67.5, 58.7. Less to fill up: [27648, 5120] m 8 49.1, 46.9,
// m 64 58.2, 60.2
static int gate_waves(int rows, int m) {
  auto fill = [&](int waves) {
    const int blocks = (rows + waves * 16 - 1) / (waves * 16);
    return (double)blocks / ((blocks + 255) / 256 * 256);
  };
  const int now = m > 16 && (rows + 127) / 128 >= 200 ? 8 : 4;
  int best = now;
  if (rows <= 4 * 256 * 64)
    for (int waves = 4; waves <= 8; ++waves)
      if (fill(waves) > fill(best) * (best != now ? 1.0 : m > 32 ? 1.2 : 1.08)) best = waves;
  return best == now ? 0 : best;
}
template <int BM>
static void gate_of_waves(const TileArgs& a, int waves) {
  if (waves == 4) launch_tile<64, BM, 4, GATED>(a);
  else if (waves == 5) launch_tile<80, BM, 4, GATED, 5>(a);
  else if (waves == 6) launch_tile<96, BM, 4, GATED, 6>(a);
  else if (waves == 7) launch_tile<112, BM, 4, GATED, 7>(a);
  else launch_tile<128, BM, 4, GATED, 8>(a);
}

template <int BN, int BM, int WN, int WB, int XB, int WAVES, int END>
static void launch_wide(const TileArgs& a) {
  const auto kernel = wide_kernel<BN, BM, WN, WB, XB, WAVES, END>;
  const int lds = MfmaTile<BN, BM, WN, WB, XB, WAVES>::LDS, per = END == GATED ? BN / 2 : BN;
  const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  TORCH_CHECK(e == hipSuccess, "no LDS for weight tiles");
  hipLaunchKernelGGL(kernel, dim3(((a.N + per - 1) / per * a.splits * ((a.m + BM - 1) / BM) + 7) / 8 * 8), dim3(WAVES * 64), lds, cur_stream(), a);
}

// Whether blocks begin at different places of k (first_step): by the weights' shape alone.
// Whole sums also over rows 4 KB apart: gate [16384, 2048] m 8 16, 13 us, m 64 17, 15
static bool turns(int K, int splits) {
  return K <= 16384 && (K % (splits > 1 ? 4096 : 2048) == 0 || (splits > 1 && K % splits == 0 && K / splits % 2048 == 0));
}

template <int END>
static void run_tile(TileArgs a) {
  a.whole = a.K / 64 / a.splits;
  a.more = a.K / 64 % a.splits;
  a.inv = 65536 / a.splits + 1;
  const int rows = END == GATED ? 2 * a.N : a.N, units = (rows + 127) / 128 * a.splits;
  a.turned = !turns(a.K, a.splits) ? 0 : gate_tile(rows, 256) == 160 ? 640 : 128;
  // Whether a die has a run of blocks, and so few parts of x, where x is larger than its L2 has
  // room for beside the weights; else blocks go round the dies, which spreads what the next
  // kernel reads. us, going round first: m 32 by [8192, 28672] 77.4, 76.3; with the norm that
  // follows, m 256 by [3584, 3584] 21.6, 25.3; [1536, 8960] 22.9, 25.8; m 192 by [3584, 18944]
  // 41.8, 43.6; [4096, 14336], whose blocks begin at different places, 40.0, 38.7; m 256
  // 46.8, 42.0; [8192, 28672] 125, 120
  const int64_t x = (int64_t)a.m * a.K;
  a.runs = END == PART ? x > (a.m <= 64 ? 2 << 19 : a.turned ? 3 << 19 : 7 << 19) : a.m > 64;
  if constexpr (END == GATED)
    if (const int waves = a.m <= 64 && !a.turned && a.splits == 1 ? gate_waves(rows, a.m) : 0)
      return a.m <= 16 ? gate_of_waves<16>(a, waves) : a.m <= 32 ? gate_of_waves<32>(a, waves) : gate_of_waves<64>(a, waves);
  if (a.m <= 16) launch_tile<64, 16, 4, END>(a);
  else if (a.m <= 32) {
    if (units >= 200) launch_tile<128, 32, 4, END>(a);
    else launch_tile<64, 32, 4, END>(a);
  } else if (a.m <= 64) {
    if (units >= 200) launch_tile<128, 64, 3, END>(a);
    else launch_tile<64, 64, 4, END>(a);
  } else if (a.K > 1 << 22) {  // from 2^23 on offsets of 256 rows take more than 32 bits
    launch_tile<128, 64, 3, END>(a);
  } else {
    if constexpr (END == GATED) {
      const int wide = gate_tile(rows, a.m);
      if (wide == 256 && a.m <= 128) return launch_wide<256, 128, 4, 4, 2, 4, END>(a);
      if (wide == 256 && a.m <= 192) return launch_wide<256, 192, 2, 3, 2, 4, END>(a);
      if (wide == 256) return launch_wide<256, 256, 2, 3, 2, 4, END>(a);
      if (wide == 160) return launch_wide<160, 256, 1, 3, 3, 4, END>(a);
    }
    if constexpr (END == GATED)
      // half as many weight rows a block while those make one round: m 80 and 128 by [16384,
      // 2048] 21 and 24 us, 18 and 19 so; [13824, 4096] 40 and 44, 31 and 35; past a round
      // they lose: [22016, 2048] 25 and 29, 30 and 34
      if (a.m <= 128 && rows <= 256 * 64) return launch_wide<64, 128, 2, 4, 3, 4, END>(a);
    if constexpr (END == PART)
      // the same of parts (parts_of): m 100 by [896, 4864] with its norm 13.5, 12.4; [1024, 1024]
      // 9.6, 8.3; in twice the parts [3584, 3584] m 100 17.8, now 15.3, m 192 21.8, 21.0, m 256 22.8,
      // 22.6 (of two blocks of 128 rows of x 23.7)
      if ((rows + 63) / 64 * a.splits <= 256 && (int64_t)rows * a.K <= 20000000) {
        if (a.m <= 128) return launch_wide<64, 128, 2, 4, 3, 4, END>(a);
        if (a.m <= 192) return launch_wide<64, 192, 2, 4, 3, 4, END>(a);
        return launch_wide<64, 256, 2, 4, 3, 8, END>(a);
      }
    if (a.m <= 128 || units < 160) {
      if (a.m <= 128 && units <= 256 && a.whole > 24) launch_wide<128, 128, 2, 4, 3, 4, END>(a);
      else launch_wide<128, 128, 4, 3, 2, 8, END>(a);
    } else if (a.m > 192) launch_wide<128, 256, 2, 3, 3, 8, END>(a);
    else if constexpr (END == GATED) launch_wide<128, 192, 2, 4, 4, 4, END>(a);
    else launch_wide<128, 192, 2, 4, 4, 8, END>(a);
  }
}

static TileArgs tile_args(const Tensor& x, const Tensor& w) {
  check_io(x, torch::kBFloat16);
  check_io(w, torch::kBFloat16);
  TileArgs a{};
  CHK(w.dim() == 2 && w.size(1) % 64 == 0 && w.size(1) > 0 && x.size(-1) == w.size(1));
  CHK(w.size(0) >= 1 && w.size(0) <= 1 << 26 && w.size(1) <= 1 << 26);
  a.K = (int)w.size(1);
  const int64_t m = x.numel() / a.K;
  CHK(m >= 1 && m <= 256);
  CHK(((size_t)x.data_ptr() & 15) == 0 && ((size_t)w.data_ptr() & 15) == 0);
  a.m = (int)m;
  a.N = (int)w.size(0);
  a.x = P<bf16_t>(x);
  a.w = P<bf16_t>(w);
  return a;
}

// Parts of k, as the rules of which products these are count them (ops.tile_splits): as few as
// give some 450 blocks of 64 weight rows, of 4 steps at least
static int splits_of(int rows, int steps) {
  const int tiles = (rows + 63) / 64;
  return std::max(1, std::min({(448 + tiles - 1) / tiles, steps / 4, 16}));
}

// What k is split in: of up to 20 10^6 weights in as many as make one round of the chip, where
// they fill it, as fewer sums are then written and read. us with the norm that reads them, splits_of
// first: m 8 [3584, 3584] 10.4, 9.9, [1536, 8960] 11.3, 10.0; m 45 [2048, 8192] 14.6, 13.0, [3072,
// 2048] 11.3, 9.3; m 128 [4096, 4096] 20.6, 17.7; m 256 [2048, 2048] 18.7, 17.7. Larger weights
// gain nothing from 65 rows on: m 8 and 192 [8192, 8192] 28.8, 28.7 and 42.6, 51.3, [4096, 14336]
// 25.6, 25.4 and 40.5, 53.7; nor do they in two thirds of a round: m 8 [6144, 4096] 14.7, 16.5.
//
// Of larger ones in one more where two blocks a CU then are all there, unless blocks of the former begin
// at different places of k (turns): 8 and 9, [3584, 18944] m 8 28.1, 27.1, m 16 29.2, 26.4, m 128
// 37.8, 36.0, m 256 51.6, 49.0; 7 and 8, [4096, 11008] m 8 22.2, 21.3, m 256 40.9, 37.2; [4096, 14336], whose 7
// turn, m 8 23.8, 23.9, m 32 24.4, 25.3, m 128 35.8, 34.1. Of 32 tiles and fewer 14 and 16 are the same
// ([2048, 11008] m 8 13.4, 13.7).
static int parts_of(int rows, int steps) {
  const int tiles = (rows + 63) / 64, n = splits_of(rows, steps), one = 256 / tiles, two = 512 / tiles;
  if (one >= 2 && one < n && one * tiles >= 200 && (int64_t)rows * steps <= 312500) return one;
  return two > n && two <= 16 && tiles > 32 && steps >= 4 * two && !turns(steps * 64, n) ? two : n;
}

static Tensor sized(const Tensor& x, int64_t n) {
  auto shape = x.sizes().vec();
  shape.back() = n;
  return torch::empty(shape, x.options());
}

// fp32 [splits, m, N]
Tensor tile_parts(Tensor x, Tensor w) {
  auto a = tile_args(x, w);
  a.splits = parts_of(a.N, a.K / 64);
  auto part = torch::empty({a.splits, a.m, a.N}, x.options().dtype(torch::kFloat32));
  a.y = part.data_ptr();
  run_tile<PART>(a);
  return part;
}

Tensor tile_linear(Tensor x, Tensor w, OptT bias) {
  auto a = tile_args(x, w);
  if (bias) {
    check_io(*bias, torch::kBFloat16);
    CHK(bias->numel() == a.N);
    a.bias = P<bf16_t>(*bias);
  }
  auto y = sized(x, a.N);
  a.splits = a.N % 4 ? 1 : parts_of(a.N, a.K / 64);
  if (a.splits == 1) {
    a.y = y.data_ptr();
    run_tile<STORE>(a);
    return y;
  }
  auto part = torch::empty({a.splits, a.m, a.N}, x.options().dtype(torch::kFloat32));
  a.y = part.data_ptr();
  run_tile<PART>(a);
  hipLaunchKernelGGL((finish_kernel<false>), dim3((a.N + 1023) / 1024, a.m), dim3(256), 0, cur_stream(),
                     part.data_ptr<float>(), a.bias, M<bf16_t>(y), a.m, a.N, a.splits);
  return y;
}

// Parts of k of the gated product: one, and no kernel that sums them up, where that leaves
// blocks enough. us, parts (and the kernel) first: [16384, 2048] m 8 15, 13, m 45 17, 14,
// m 128 23, 19; [9728, 896] m 8 8, 7, m 64 13, 8, m 256 23, 13; [13824, 4096] m 8 25, 22, m 64
// 36, 27; [22016, 2048] m 16 22, 20, m 256 50, 33. Fewer blocks and longer sums lose: [8192,
// 4096] m 8 17, 23; [14336, 8192] m 8 42, 44, m 160 62, 74; and so do tiles that just pass
// one round: [17920, 4096] m 32 40, 38, m 160 62, 76.
// (ops.gate_splits says the same)
static int gate_splits(int rows, int steps) {
  const int tiles = (rows + 63) / 64;
  if (steps <= 16 || (tiles >= 160 && steps <= (tiles > 256 && tiles < 320 ? 32 : 96))) return 1;
  return parts_of(rows, steps);
}

Tensor tile_swiglu(Tensor x, Tensor w) {
  auto a = tile_args(x, w);
  CHK(a.N % 8 == 0);
  const int I = a.N / 2;
  auto y = sized(x, I);
  a.splits = gate_splits(a.N, a.K / 64);
  if (a.splits == 1) {
    a.N = I;
    a.y = y.data_ptr();
    run_tile<GATED>(a);
    return y;
  }
  auto part = torch::empty({a.splits, a.m, a.N}, x.options().dtype(torch::kFloat32));
  a.y = part.data_ptr();
  run_tile<PART>(a);
  hipLaunchKernelGGL((finish_kernel<true>), dim3((I + 1023) / 1024, a.m), dim3(256), 0, cur_stream(),
                     part.data_ptr<float>(), nullptr, M<bf16_t>(y), a.m, I, a.splits);
  return y;
}

// (h, norm(h) w) with h = x + sum of the parts; w none: h alone
std::vector<Tensor> parts_add_norm(Tensor part, Tensor x, OptT w, double eps, double add, bool round) {
  check_io(part, torch::kFloat32);
  check_io(x, torch::kBFloat16);
  CHK(part.dim() == 3 && part.numel() == x.numel() * part.size(0) && part.size(2) == x.size(-1));
  const int D = (int)x.size(-1), m = (int)part.size(1);
  CHK(D % 4 == 0 && D <= 16384 && ((size_t)x.data_ptr() & 7) == 0);
  auto h = torch::empty_like(x);
  Tensor n;
  const bf16_t* wp = nullptr;
  if (w) {
    check_io(*w, torch::kBFloat16);
    CHK(w->numel() == D && ((size_t)w->data_ptr() & 7) == 0);
    n = torch::empty_like(x);
    wp = P<bf16_t>(*w);
  }
  bf16_t* np = w ? M<bf16_t>(n) : nullptr;
#define GO(NC_, T_) hipLaunchKernelGGL((add_norm_kernel<NC_, T_>), dim3(m), dim3(T_), 0, cur_stream(), part.data_ptr<float>(), \
                                       P<bf16_t>(x), wp, M<bf16_t>(h), np, m, D, (int)part.size(0), (float)eps, (float)add, round)
  if (D <= 1024) GO(1, 256);
  else if (D <= 2048) GO(1, 512);
  else if (D <= 4096) GO(1, 1024);
  else if (D <= 8192) GO(2, 1024);
  else GO(4, 1024);
#undef GO
  if (w) return {h, n};
  return {h};
}

// What follows a layer's attention, in one call from Python, which a short prompt through a
// small model waits for: h = x + heads Wo^T, its norm, the gated activation, h + that Wd^T,
// and the next layer's norm of it (`after`; none: the stream alone)
std::vector<Tensor> tile_rest(Tensor heads, Tensor wo, Tensor x, Tensor post, double post_eps, Tensor gate_up, Tensor down,
                              OptT after, double after_eps) {
  auto mid = parts_add_norm(tile_parts(heads, wo), x, post, post_eps, 0.0, false);
  return parts_add_norm(tile_parts(tile_swiglu(mid[1], gate_up), down), mid[0], after, after_eps, 0.0, after.has_value());
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("tile_rest", &tile_rest);
  m.def("tile_splits", [](int64_t n, int64_t k) { return splits_of((int)n, (int)(k / 64)); });
  m.def("parts_of", [](int64_t n, int64_t k) { return parts_of((int)n, (int)(k / 64)); });
  m.def("gate_waves", [](int64_t rows, int64_t m) { return gate_waves((int)rows, (int)m); });
  m.def("gate_splits", [](int64_t n, int64_t k) { return gate_splits((int)n, (int)(k / 64)); });
  m.def("gate_tile", [](int64_t rows, int64_t m) { return gate_tile((int)rows, (int)m); });
  m.def("tile_parts", &tile_parts);
  m.def("tile_linear", &tile_linear);
  m.def("tile_swiglu", &tile_swiglu);
  m.def("parts_add_norm", &parts_add_norm);
}
