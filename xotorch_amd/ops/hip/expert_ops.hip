// CDNA4 (gfx950) kernels of sparse feed-forwards: a mixture of small experts,
// routed and computed without the host seeing a count.
//   - router: logits on matrix cores (fp32 accumulation), sigmoid scores, a
//     correction that only chooses, group-limited top-k, or a softmax over the
//     chosen logits; experts that every token uses, gated or not; counts per block
//   - place: every (token, expert) pair gets a row; rows of an expert lie
//     together, in token order
//   - grouped products: gate and up of a pair's token with the gated activation
//     in the epilogue, or up alone, squared where it is positive, then down; a
//     weight-streaming form for few tokens per expert and a tiled form for many.
//     A weight that multiplies a pair's input scales the product's rows
//   - add_norm: stream += mult * (a sublayer's output, or the weighted sum of a
//     token's expert rows), then the stream's norm for the next sublayer
//
// Two element types: bf16 and fp32 (fp32 MFMA throughout).

#include "common.h"
#include "stream_tile.h"

// ---------------------------------------------------------------------------
// router
// ---------------------------------------------------------------------------

constexpr int RT = 16;          // tokens of a router block
constexpr int FEW_BLOCKS = 16;  // of the router, whose counts need no kernel of their own to be scanned
constexpr int MAX_EXPERTS = 512, MAX_PICK = 16;  // shared ones among the experts

// pick of E experts are chosen, then come top - pick that every token uses, all
// in all; tile: rows of a tile
// gate: the weight of these is the sigmoid of one more row of w, else one
// narrow: logits as bf16, as a linear of their own leaves them; given: x are the logits
struct RouteArgs { int T, D, E, top, groups, keep, nblk, tile; float scale; int pick, all, softmax, gate, narrow, given; };

// RW waves share k. Sixteen lanes choose for a token, J experts each.
template <typename T, bool WHOLE, int J, int RW>
__global__ __launch_bounds__(64 * RW) void route_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ correction, int* __restrict__ idx,
    float* __restrict__ weight, int* __restrict__ rank, int* __restrict__ counts, RouteArgs a) {
  typedef Frag<T> F;
  extern __shared__ float lds[];  // choice, scores [RT][E]; partial sums [RW][RT][65]; chosen [RT][top]; open [RT]
  float* choice = lds;
  float* score = choice + RT * a.E;
  float* part = score + RT * a.E;
  int* chosen = (int*)(part + RW * RT * 65);
  float* open = (float*)(chosen + RT * a.top);  // [RT], the gate of the experts that every token uses
  const int Z = a.E + a.gate;
  const int t0 = blockIdx.x * RT, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
  const T* xr = x + (size_t)min(t0 + col, a.T - 1) * a.D;
  const int steps = (a.D + F::K - 1) / F::K;
  auto scored = [&](int t, int e, float z) {  // logit e of token t
    const float s = a.softmax && e < a.E ? z : 1.f / (1.f + expf(-z));
    if (e < a.E) {
      score[t * a.E + e] = s;
      choice[t * a.E + e] = correction ? s + ld(correction + e) : s;
    } else open[t] = s;
  };
  if (a.given) {
    for (int i = threadIdx.x; i < RT * a.E; i += 64 * RW) {
      const int t = i / a.E, e = i - t * a.E;
      scored(t, e, ld(x + (size_t)min(t0 + t, a.T - 1) * a.E + e));
    }
    __syncthreads();
  }
  for (int e0 = 0; e0 < Z && !a.given; e0 += 64) {
    floatx4 acc[4];
    const T* wr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i] = (floatx4)(0.f);
      wr[i] = w + (size_t)min(e0 + i * 16 + col, Z - 1) * a.D;
    }
    auto run = [&](int c, auto count) {  // `count` steps from c on, loads first
      constexpr int UN = decltype(count)::value;
      typename F::V xf[UN], wf[UN][4];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int k = (c + u) * F::K + quad * F::PER;
        xf[u] = ld_frag<T, WHOLE>(xr, k, a.D);
#pragma unroll
        for (int i = 0; i < 4; ++i) wf[u][i] = ld_frag<T, WHOLE>(wr[i], k, a.D);
      }
#pragma unroll
      for (int u = 0; u < UN; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = mma(wf[u][i], xf[u], acc[i]);
    };
    int c = wave * 4;
    for (; c + 4 <= steps; c += 4 * RW) run(c, std::integral_constant<int, 4>());
    for (; c < steps; ++c) run(c, std::integral_constant<int, 1>());
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[(wave * RT + col) * 65 + i * 16 + quad * 4 + r] = acc[i][r];
    __syncthreads();
    for (int i = threadIdx.x; i < RT * 64; i += 64 * RW) {
      const int t = i >> 6, e = e0 + (i & 63);
      if (e < Z) {
        float z = 0.f;
#pragma unroll
        for (int v = 0; v < RW; ++v) z += part[(v * RT + t) * 65 + (i & 63)];
        scored(t, e, a.narrow ? rounded(z) : z);
      }
    }
    __syncthreads();
  }
  const int size = a.E / a.groups;
  const int t = threadIdx.x >> 4, l = threadIdx.x & 15;
  if (t < RT) {  // rows of LDS are the sixteen lanes' own
    float* ch = choice + t * a.E;
    if (a.keep < a.groups) {
      // lane l (and l + 16, ..) scores group l by its two best
      float* gs = part + t * a.groups;
      for (int g = l; g < a.groups; g += 16) {
        float b1 = -INFINITY, b2 = -INFINITY;
#pragma unroll 4
        for (int i = 0; i < size; ++i) {
          const float v = ch[g * size + i];
          b2 = fmaxf(b2, fminf(v, b1));
          b1 = fmaxf(b1, v);
        }
        gs[g] = size > 1 ? b1 + b2 : b1;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (int g = l; g < a.groups; g += 16) {
        const float mine = gs[g];
        int better = 0;
        for (int o = 0; o < a.groups; ++o) better += gs[o] > mine || (gs[o] == mine && o < g);
        if (better >= a.keep)
          for (int i = 0; i < size; ++i) ch[g * size + i] = -INFINITY;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    float v[J];
#pragma unroll
    for (int j = 0; j < J; ++j) v[j] = l + j * 16 < a.E ? ch[l + j * 16] : -INFINITY;
    const bool valid = t0 + t < a.T;
    float mine = 0.f;  // score of the choice that lane l weighs
    for (int k = 0; k < a.pick; ++k) {
      float best = v[0];
#pragma unroll
      for (int j = 1; j < J; ++j) best = fmaxf(best, v[j]);
      best = row_max(best);
      int at = INT_MAX;
#pragma unroll
      for (int j = J - 1; j >= 0; --j)
        if (v[j] == best) at = l + j * 16;
      at = min(row_min(at), a.E - 1);  // the lowest of equals
#pragma unroll
      for (int j = 0; j < J; ++j)
        if (at == l + j * 16) v[j] = -INFINITY;
      if (l == k) mine = score[t * a.E + at];
      if (l == 0) {
        chosen[t * a.top + k] = valid ? at : -1;
        if (valid) idx[(size_t)(t0 + t) * a.top + k] = at;
      }
    }
    if (a.softmax) {
      const float e = l < a.pick ? expf(mine - row_max(l < a.pick ? mine : -INFINITY)) : 0.f;
      mine = e / row_sum(e);
    }
    if (valid && l < a.pick) weight[(size_t)(t0 + t) * a.top + l] = mine * a.scale;
    for (int k = a.pick + l; k < a.top; k += 16) {
      const int e = a.E + k - a.pick;
      chosen[t * a.top + k] = valid ? e : -1;
      if (valid) {
        idx[(size_t)(t0 + t) * a.top + k] = e;
        weight[(size_t)(t0 + t) * a.top + k] = a.gate ? open[t] : 1.f;
      }
    }
  }
  __syncthreads();
  // place among the block's pairs of the same expert, and the block's counts;
  // chosen holds RT * top entries, a multiple of four
  const int4* four = (const int4*)chosen;
  const int pairs = (min(RT, a.T - t0) * a.top + 3) >> 2;  // fours of them
  for (int e = threadIdx.x; e < a.all; e += 64 * RW) {
    int n = 0;
    int* dst = rank + (size_t)t0 * a.top;
    for (int o = 0; o < pairs; ++o) {
      const int4 c = four[o];
      if (c.x == e) dst[o * 4] = n++;
      if (c.y == e) dst[o * 4 + 1] = n++;
      if (c.z == e) dst[o * 4 + 2] = n++;
      if (c.w == e) dst[o * 4 + 3] = n++;
    }
    counts[(size_t)e * a.nblk + blockIdx.x] = n;
  }
}

// counts [E][nblk] -> exclusive sums along nblk, in place, and the totals [E]
__global__ __launch_bounds__(256) void count_scan_kernel(int* __restrict__ counts, int* __restrict__ total, int nblk) {
  __shared__ int sums[256];
  int* row = counts + (size_t)blockIdx.x * nblk;
  const int per = (nblk + 255) / 256, lo = threadIdx.x * per, hi = min(lo + per, nblk);
  int n = 0;
  for (int i = lo; i < hi; ++i) n += row[i];
  sums[threadIdx.x] = n;
  __syncthreads();
  for (int d = 1; d < 256; d <<= 1) {
    const int o = threadIdx.x >= d ? sums[threadIdx.x - d] : 0;
    __syncthreads();
    sums[threadIdx.x] += o;
    __syncthreads();
  }
  int at = sums[threadIdx.x] - n;
  for (int i = lo; i < hi; ++i) {
    const int c = row[i];
    row[i] = at;
    at += c;
  }
  if (threadIdx.x == 255) total[blockIdx.x] = sums[255];
}

// Rows of all pairs: row[pair], token[row] and, by_row given, the pair's weight;
// first row of every expert [E + 1]; tiles (expert, first row), expert -1 past
// the last, and behind them (-1, how many there are).
__global__ __launch_bounds__(256) void place_kernel(
    const int* __restrict__ idx, const int* __restrict__ rank, const int* __restrict__ before,
    const int* __restrict__ total, const float* __restrict__ weight, int* __restrict__ row, int* __restrict__ token,
    float* __restrict__ by_row, int* __restrict__ first, int2* __restrict__ tiles, int max_tiles, RouteArgs a) {
  __shared__ int at[MAX_EXPERTS], cnt[MAX_EXPERTS], tile_at[MAX_EXPERTS], ends[2];
  // few blocks of the router need no scan (route): their counts are added up here
  const bool few = a.nblk <= FEW_BLOCKS;
  for (int e = threadIdx.x; e < a.all; e += 256) {
    int n = 0;
    if (few)
      for (int i = 0; i < a.nblk; ++i) n += before[(size_t)e * a.nblk + i];
    cnt[e] = few ? n : total[e];
  }
  __syncthreads();
  if (threadIdx.x < 64) {  // one wave scans, E/64 each
    const int per = (a.all + 63) / 64, lo = threadIdx.x * per, hi = min(lo + per, a.all);
    int n = 0, m = 0;
    for (int e = lo; e < hi; ++e) { n += cnt[e]; m += (cnt[e] + a.tile - 1) / a.tile; }
    int sn = n, sm = m;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int on = __shfl_up(sn, d), om = __shfl_up(sm, d);
      if (threadIdx.x >= d) { sn += on; sm += om; }
    }
    if (threadIdx.x == 63) { ends[0] = sn; ends[1] = sm; }
    sn -= n;
    sm -= m;
    for (int e = lo; e < hi; ++e) {
      at[e] = sn;
      tile_at[e] = sm;
      sn += cnt[e];
      sm += (cnt[e] + a.tile - 1) / a.tile;
    }
  }
  __syncthreads();
  const int pair = blockIdx.x * 256 + threadIdx.x;
  if (pair < a.T * a.top) {
    const int e = idx[pair], t = pair / a.top;
    int r = at[e] + rank[pair];
    if (few)
      for (int i = 0; i < t / RT; ++i) r += before[(size_t)e * a.nblk + i];
    else r += before[(size_t)e * a.nblk + t / RT];
    row[pair] = r;
    token[r] = t;
    if (by_row) by_row[r] = weight[pair];
  }
  if (blockIdx.x) return;
  for (int e = threadIdx.x; e < a.all; e += 256) {
    first[e] = at[e];
    for (int i = 0; i * a.tile < cnt[e]; ++i) tiles[tile_at[e] + i] = make_int2(e, at[e] + i * a.tile);
  }
  for (int i = ends[1] + threadIdx.x; i < max_tiles; i += 256) tiles[i] = make_int2(-1, 0);
  if (threadIdx.x == 0) {
    first[a.all] = ends[0];
    tiles[max_tiles] = make_int2(-1, ends[1]);
  }
}

// ---------------------------------------------------------------------------
// grouped products
// ---------------------------------------------------------------------------

struct Act { float alpha, limit, plus; };
// min(g, limit) sigmoid(alpha min(g, limit)) (clamp(u, -limit, limit) + plus)
DEVINL float gated(float g, float u, const Act& a) {
  g = fminf(g, a.limit);
  u = fminf(fmaxf(u, -a.limit), a.limit);
  return g * sigmoidf(a.alpha * g) * (u + a.plus);
}

// What a product is: of a pair's own row; of its token with gate and up weights
// and the gated activation; of its token with one set of weights and the square
// of what is positive; of its token with gate and up weights and silu (no limits); the
// same where there is but one expert, of all rows.
enum Product { PLAIN, GATED, RELU2, SWIGLU, DENSE };
constexpr bool has_gate(int kind) { return kind == GATED || kind == SWIGLU || kind == DENSE; }
constexpr bool of_own_row(int kind) { return kind == PLAIN || kind == DENSE; }

struct GroupArgs {
  int K, kp, F, E;  // valid and stored length of a weight row, output features, experts
  int xs, ys;       // row strides of input and output
};

// A product's rows times what scales them, through its activation
template <int KIND>
DEVINL float activated(float by, float g, float u, const Act& a) {
  if (KIND == GATED) return gated(by * g, by * u, a);
  if (KIND == SWIGLU || KIND == DENSE) return siluf(by * g) * (by * u);
  g = by * g;
  if (KIND == RELU2) g = fmaxf(g, 0.f) * g;
  return g;
}

// Few tokens per expert: a block owns 16 output features of one expert; its
// four waves split k and walk the expert's rows up to 64 (GATED: 32) at a time. GATED:
// weights [E][2][F][kp]; else [E][F][kp]. Input rows are gathered by token but
// for PLAIN. by_row: what the rows of the product are scaled with.
template <typename T, int KIND, bool WHOLE>
__global__ __launch_bounds__(256) void expert_stream_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const int* __restrict__ first, const int* __restrict__ token,
    const float* __restrict__ by_row, T* __restrict__ y, GroupArgs a, Act act) {
  typedef Frag<T> F;
  constexpr int NW = has_gate(KIND) ? 2 : 1, MOST = 4 / NW;
  __shared__ float part[4][NW][MOST * 16][17];
  // the last experts are the ones that every token uses: the longest come first
  const int e = gridDim.y - 1 - blockIdx.y, f0 = blockIdx.x * 16;
  const int lo = first[e], hi = first[e + 1];
  if (lo == hi) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
  const T* wr[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) wr[i] = w + (((size_t)e * NW + i) * a.F + f0 + col) * a.kp + quad * F::PER;
  const int steps = (a.K + F::K - 1) / F::K;
  auto round = [&](int r0, auto tiles) {  // 16 * MT rows
    constexpr int MT = decltype(tiles)::value, UN = MT == 4 ? 4 : 8 / NW;
    floatx4 acc[NW][MT];
    const T* xr[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int r = min(r0 + m * 16 + col, hi - 1);
      xr[m] = x + (size_t)(KIND == PLAIN ? r : token[r]) * a.xs;
#pragma unroll
      for (int i = 0; i < NW; ++i) acc[i][m] = (floatx4)(0.f);
    }
    auto run = [&](int c, auto count) {  // `count` steps from c on, loads first
      constexpr int N = decltype(count)::value;
      typename F::V wf[N][NW], xf[N][MT];
#pragma unroll
      for (int u = 0; u < N; ++u) {
#pragma unroll
        for (int i = 0; i < NW; ++i) wf[u][i] = *(const typename F::V*)(wr[i] + (size_t)(c + u) * F::K);
#pragma unroll
        for (int m = 0; m < MT; ++m) xf[u][m] = ld_frag<T, WHOLE>(xr[m], (c + u) * F::K + quad * F::PER, a.K);
      }
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int i = 0; i < NW; ++i) acc[i][m] = mma(wf[u][i], xf[u][m], acc[i][m]);
    };
    int c = wave * UN;
    for (; c + UN <= steps; c += 4 * UN) run(c, std::integral_constant<int, UN>());
    for (; c < steps; ++c) run(c, std::integral_constant<int, 1>());
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wave][i][m * 16 + col][quad * 4 + r] = acc[i][m][r];
    __syncthreads();
    const int n = min(16 * MT, hi - r0);
    for (int i = threadIdx.x; i < n * 16; i += 256) {
      const int t = i >> 4, f = i & 15;
      float v[NW];
#pragma unroll
      for (int j = 0; j < NW; ++j)
        v[j] = part[0][j][t][f] + part[1][j][t][f] + part[2][j][t][f] + part[3][j][t][f];
      const float by = KIND != PLAIN && by_row ? by_row[r0 + t] : 1.f;
      st(y + (size_t)(r0 + t) * a.ys + f0 + f, activated<KIND>(by, v[0], v[NW - 1], act));
    }
    __syncthreads();
  };
  int r0 = lo;
  for (; hi - r0 > 32; r0 += MOST * 16) round(r0, std::integral_constant<int, MOST>());
  if (hi - r0 > 16) round(r0, std::integral_constant<int, 2>());
  else if (hi > r0) round(r0, std::integral_constant<int, 1>());
}

// Many tokens per expert (bf16): up to TOK tokens x BN weight rows (GATED: BN / 2 gate and
// the same of up) per block, by mfma_tile.h. What bounds them is the matrix cores, and
// rows of a tile that no token fills: an expert's rows go over its tiles evenly, in steps
// of 32. 8 experts of 4096 x 14336, two of them a token, both products, us: 2100 tokens 1340
// (in steps of 64 by eight waves 1480), 1500 939 (1069), 1000 776 (855), 500 560 (598), 300 538
// (557). Up to 700 tokens the weights bound them, at some 4.5 TB/s.

// Where an expert's weight rows lie: in one tensor, or in one tensor each
struct Stacked {
  const bf16_t* w;
  DEVINL const bf16_t* of(int e, size_t expert) const { return w + e * expert; }
};
constexpr int MOST_LISTED = 256;
struct Listed {
  const bf16_t* w[MOST_LISTED];
  DEVINL const bf16_t* of(int e, size_t) const { return w[e]; }
};

// Waves along the weight rows, buffers of weights and tokens
template <int BN, int BM, int WN_, int WB, int XB> struct Shape : MfmaTile<BN, BM, WN_, WB, XB> { static constexpr int WN = WN_; };
template <int BN, int BM> struct ExpertTile;
template <> struct ExpertTile<256, 64> : Shape<256, 64, 4, 4, 4> {};
template <> struct ExpertTile<256, 128> : Shape<256, 128, 2, 3, 3> {};
template <> struct ExpertTile<256, 160> : Shape<256, 160, 2, 3, 3> {};
template <> struct ExpertTile<256, 192> : Shape<256, 192, 2, 3, 2> {};
template <> struct ExpertTile<256, 224> : Shape<256, 224, 2, 3, 2> {};
template <> struct ExpertTile<256, 256> : Shape<256, 256, 2, 3, 2> {};
template <> struct ExpertTile<128, 64> : Shape<128, 64, 2, 3, 3> {};
template <> struct ExpertTile<128, 128> : Shape<128, 128, 2, 3, 2> {};
template <> struct ExpertTile<128, 192> : Shape<128, 192, 2, 4, 4> {};
template <> struct ExpertTile<128, 256> : Shape<128, 256, 2, 3, 3> {};
// of all forms that a kernel of BN weight rows and TOK tokens may take
template <int BN, int TOK> constexpr int expert_lds() {
  int most = std::max(ExpertTile<BN, 64>::LDS, ExpertTile<BN, 128>::LDS);
  if constexpr (TOK == 256)  // and of 128 weight rows
    most = std::max({most, expert_lds<128, 128>(), ExpertTile<128, 192>::LDS, ExpertTile<128, 256>::LDS, ExpertTile<256, 160>::LDS,
                     ExpertTile<256, 192>::LDS, ExpertTile<256, 224>::LDS, ExpertTile<256, 256>::LDS});
  return most;
}

// One tile: tokens r0 up to hi, of which there are at most BM. TAIL: rows of x may end within
// a step; FAR: x takes 4 GB or more
template <int KIND, int BN, int BM, bool TAIL, bool FAR>
DEVINL void expert_tile(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const int* __restrict__ token,
                        const float* __restrict__ by_row, bf16_t* __restrict__ y, const GroupArgs& a, const Act& act,
                        int r0, int hi, int fb, bf16_t* buf) {
  typedef ExpertTile<BN, BM> Sh;
  constexpr bool TWO = has_gate(KIND), OWN = of_own_row(KIND);  // TWO: weight rows are gate and up
  constexpr int R = Sh::R, C = Sh::C, ROWS = R * 16;  // a wave's weight rows: gate rows, then the same of up
  constexpr int WL = Sh::WL, XL = Sh::XL;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
  const int wf = wave % Sh::WN, wt = wave / Sh::WN, f0 = fb * (TWO ? BN / 2 : BN);
  const int piece = ((lane & 7) ^ (lane >> 3)) * 8, up = TWO ? wave >> 1 : 0;  // two waves load gates, two up
  const bf16_t *wsrc = w + ((size_t)up * a.F + f0) * a.kp, *xsrc = OWN ? x + (size_t)r0 * a.xs : x;
  unsigned woff[WL], wto[WL], xoff[XL];
  const char* xfar[FAR ? XL : 1];
#pragma unroll
  for (int i = 0; i < WL; ++i) {  // F % 16 == 0: the 8 rows of a load are there, or none of them
    const int r = ((TWO ? wave & 1 : wave) * WL + i) * 8;
    woff[i] = ((unsigned)(min(r, a.F - 8 - f0) + (lane >> 3)) * a.kp + piece) * 2;
    wto[i] = (TWO ? r / (ROWS / 2) * ROWS + up * (ROWS / 2) + r % (ROWS / 2) : r) * 128;
  }
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int t = min(r0 + (wave * XL + i) * 8 + (lane >> 3), hi - 1);
    if constexpr (FAR) xfar[i] = (const char*)(x + (size_t)token[t] * a.xs);
    else xoff[i] = ((unsigned)(OWN ? t - r0 : token[t]) * a.xs + (TAIL ? 0 : piece)) * 2;
  }
  const int steps = (a.K + 63) / 64;
  auto stepw = [&](int s) { return StepSource(wsrc, s * 128, steps - s); };
  auto stepx = [&](int s) { return StepSource(xsrc, s * 128, steps - s); };
  auto loadw = [&](auto number, const StepSource& from, unsigned at) {
    constexpr int i = decltype(number)::value;
    from.load(woff[i], (char*)buf + at + wto[i]);
  };
  auto loadx = [&](auto number, StepSource from, unsigned at) {
    constexpr int i = decltype(number)::value;
    char* to = (char*)buf + at + (wave * XL + i) * 1024;
    // past the end of a row the weights are zero; any number of the row will do
    const int k = from.at / 2 + piece, in = TAIL && k >= a.K ? 0 : k * 2;
    if constexpr (FAR) __builtin_amdgcn_global_load_lds((glb_void*)(xfar[i] + in), (lds_void*)to, 16, 0, 0);
    else if constexpr (TAIL) {
      from.at = 0;
      from.load(xoff[i] + in, to);
    } else from.load(xoff[i], to);
  };
  floatx4 acc[R][C];
  const unsigned base = (unsigned)(size_t)(lds_void*)buf;
  walk<Sh>(acc, RowFrags<R>(base, wf * ROWS, lane), RowFrags<C>(base + Sh::XAT, wt * C * 16, lane), steps, stepw, loadw, stepx, loadx);
  constexpr int N = TWO ? R / 2 : R;
  const RowsOut<bf16_t, N * 16> rows(buf, wave, lane);
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int t0 = r0 + (wt * C + j) * 16;
    const float by = !OWN && by_row ? by_row[min(t0 + col, hi - 1)] : 1.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      ushort4_t v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = f2b(activated<KIND>(by, acc[i][j][r], acc[(i + R / 2) % R][j][r], act));
      rows.put(col, i * 16 + quad * 4, v);
    }
    rows.out([&](int r, int f, floatx4 v) {
      const int to = f0 + wf * 16 * N + f;
      if (t0 + r < hi && to < a.F) *(floatx4*)(y + (size_t)(t0 + r) * a.ys + to) = v;
    });
  }
}

constexpr int DIE_CUS = 32;  // of one of the eight dies

// Most rows of a tile, how many tiles that makes of all experts' rows, and where this lane's
// experts end among them
struct Plan { int most, tiles, end; };
DEVINL int tiles_of(unsigned rows, int most) {
  return most == 256 ? (rows + 255) / 256 : most == 192 ? (rows + 191) / 192 : (rows + 127) / 128;
}
// Where blocks are few (launch_tiles), what the last round of them leaves idle counts for more
// than what smaller tiles cost: 256, 192 or 128 rows, by the time that the rounds take, of
// which a block of n rows takes 0.4 + 0.00375 n, cut in two 0.62 of that (rows as they are shared
// out, not as the form that takes them has: gate_product's plan rounds to 32). All blocks find
// the same. us of the down product of 8 experts of 4096 x 14336, two of them a token, with 256
// and so: 2100 tokens 486, 443; 1000 tokens 305, 246; 1500 and 700, which stay with 256, 301
// and 214.
DEVINL Plan plan_of(const int* __restrict__ first, int E, int nf, int lane) {
  const int per = (E + 63) / 64, e0 = min(lane * per, E), e1 = min(e0 + per, E);
  int found = 0, tiles = 0, end = 0;
  float least = 0.f;
#pragma unroll
  for (int most : {256, 192, 128}) {
    int mine = 0;
    float tall = 0.f;
    for (int e = e0; e < e1; ++e) {
      const int rows = first[e + 1] - first[e], n = tiles_of(rows, most);
      mine += n;
      if (n) tall = fmaxf(tall, (float)rows / (float)n);
    }
    int sum = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int other = __shfl_up(sum, d);
      if (lane >= d) sum += other;
      tall = fmaxf(tall, __shfl_xor(tall, d));
    }
    const int all = __shfl(sum, 63);
    const unsigned blocks = all * nf, left = blocks % 256;
    const float each = 0.4f + 0.00375f * (float)first[E] / (float)max(all, 1), last = 0.4f + 0.00375f * tall;
    const float time = (float)(blocks / 256) * each + (left == 0 ? 0.f : left <= 128 ? 0.62f * last : last);
    if (most == 256 || time < 0.97f * least) found = most, tiles = all, end = sum, least = time;
  }
  return {found, tiles, end};
}

// The router's tiles, of which there are as many as the last of `tiles` says, or (replan) those
// of plan_of; DENSE: max_tiles of rows_of_all rows
template <int KIND, int BN, int TOK, bool FAR, typename W>
__global__ __launch_bounds__(256) void expert_tile_kernel(
    const bf16_t* __restrict__ x, W w, const int* __restrict__ first,
    const int* __restrict__ token, const int2* __restrict__ tiles, const float* __restrict__ by_row,
    bf16_t* __restrict__ y, int max_tiles, int group, int rows_of_all, bool replan, GroupArgs a, Act act) {
  extern __shared__ __attribute__((aligned(16))) bf16_t buf[];
  // blocks go round the eight dies: a die has a run of them, in panels of `group` tiles
  // whose weight rows come one after the other, so that its L2 serves both operands
  constexpr bool TWO = has_gate(KIND);
  constexpr int WIDE = TWO ? BN / 2 : BN;
  constexpr bool CUT = BN == 256 && TOK == 256;  // (up to 128 tokens gain nothing)
  const int nf = (a.F + WIDE - 1) / WIDE, lane = threadIdx.x & 63;
  Plan plan{TOK, 0, 0};
  if constexpr (KIND == DENSE) plan.tiles = max_tiles;
  else if (CUT && replan) {
    plan = plan_of(first, a.E, nf, lane);
    plan.most = __builtin_amdgcn_readfirstlane(plan.most);
    plan.tiles = __builtin_amdgcn_readfirstlane(plan.tiles);
    group = __builtin_amdgcn_readfirstlane(first[a.E]) / (a.E * plan.most) + 1;
  } else plan.tiles = __builtin_amdgcn_readfirstlane(tiles[max_tiles].y);
  const int real = plan.tiles, die = blockIdx.x & 7, each = real * nf / 8, rest = real * nf % 8, all = each + (die < rest);
  // what no more than half of a die's 32 CUs would have left to do is cut in two: 384 blocks
  // of the down product of 2100 tokens 578 us, so 522
  const int whole = CUT && all % DIE_CUS <= DIE_CUS / 2 ? all - all % DIE_CUS : all;
  int at = blockIdx.x >> 3, half = -1;
  if (at >= whole) {
    half = (at - whole) & 1;
    at = whole + ((at - whole) >> 1);
  }
  if (at >= all) return;
  const int n = die * each + min(die, rest) + at, per = group * nf, panel = n / per, in = n % per;
  const int wide = min(group, real - panel * group), m = panel * group + in % wide, fb = in / wide;
  int e = 0, lo = 0, end = rows_of_all, nth = m;
  if constexpr (KIND != DENSE) {
    if (CUT && replan) {
      // the first lane whose experts' tiles end behind m, and its expert
      const int owner = __popcll(__ballot(plan.end <= m)), of_lane = (a.E + 63) / 64;
      nth = m - (owner ? __builtin_amdgcn_readlane(plan.end, owner - 1) : 0);
      for (e = owner * of_lane;; ++e) {
        lo = __builtin_amdgcn_readfirstlane(first[e]), end = __builtin_amdgcn_readfirstlane(first[e + 1]);
        const int tiles_here = tiles_of(end - lo, plan.most);
        if (nth < tiles_here || e + 1 >= a.E) break;
        nth -= tiles_here;
      }
    } else {
      const int2 tile = tiles[m];
      e = __builtin_amdgcn_readfirstlane(tile.x);
      lo = __builtin_amdgcn_readfirstlane(first[e]), end = __builtin_amdgcn_readfirstlane(first[e + 1]);
      nth = (__builtin_amdgcn_readfirstlane(tile.y) - lo) / TOK;
    }
  }
  // an expert's rows go over its tiles evenly, in steps of 32
  const int of = KIND == DENSE ? max_tiles : CUT ? tiles_of(end - lo, plan.most) : (end - lo + TOK - 1) / TOK, share = ((end - lo + of - 1) / of + 31) / 32 * 32;
  const int r0 = lo + nth * share, hi = min(end, r0 + share), rows = hi - r0;
  const bf16_t* we = w.of(e, (size_t)(TWO ? 2 : 1) * a.F * a.kp);
  constexpr bool TAIL = std::is_same<W, Stacked>::value && KIND != DENSE;
  auto go = [&](auto weights, auto most) {
    constexpr int N = decltype(weights)::value, M = decltype(most)::value;
    expert_tile<KIND, N, M, TAIL, FAR>(x, we, token, by_row, y, a, act, r0, hi, N == BN ? fb : fb * 2 + half, buf);
  };
  typedef std::integral_constant<int, BN> All;
  if constexpr (CUT) {
    if (half >= 0) {
      typedef std::integral_constant<int, 128> Half;
      if ((fb * 2 + half) * (WIDE / 2) >= a.F) return;
      if (rows <= 64) go(Half(), std::integral_constant<int, 64>());
      else if (rows <= 128) go(Half(), std::integral_constant<int, 128>());
      else if (rows <= 192) go(Half(), std::integral_constant<int, 192>());
      else go(Half(), std::integral_constant<int, 256>());
      return;
    }
  }
  if (rows <= 64) go(All(), std::integral_constant<int, 64>());
  else if (rows <= 128) go(All(), std::integral_constant<int, 128>());
  else if constexpr (TOK == 256) {
    if (rows <= 160) go(All(), std::integral_constant<int, 160>());
    else if (rows <= 192) go(All(), std::integral_constant<int, 192>());
    else if (rows <= 224) go(All(), std::integral_constant<int, 224>());
    else go(All(), std::integral_constant<int, 256>());
  }
}

// Few tokens (bf16, one weight tensor per expert; SWIGLU or PLAIN): a block owns BN weight rows of one of the
// router's tiles and takes its rows, up to 128, by 64 and, the last, 32 or 16. Weights bound it: they stream
// through LDS (stream_tile.h), of experts that have a row only, at 6.5 TB/s where all have. us of a whole
// sparse feed-forward in a graph, as it was, with every expert over room for all tokens from copies in
// fragment order and kernels for logits, choice, places, gathering and the activation, and so: 8 experts of 4096 x 14336, two
// of them a token: 1 token 501, 157; 2 505, 210; 8 504, 400; 32 503, 438; 128 633, 460; 128 of 2048 x 768, eight of them: 1
// token 272, 46; 8 270, 110; 32 271, 200; 128 364, 228; errors against 64 bits 0.0036 to 0.0061, 0.0023
// to 0.0025.
template <int BN, int BM> struct FewTile : TileShape<BN, BM, BM == 64 ? 3 : 4> {};
template <int BN> constexpr int few_lds() { return std::max({FewTile<BN, 16>::LDS, FewTile<BN, 32>::LDS, FewTile<BN, 64>::LDS}); }
template <int KIND, int BN, int BM>
DEVINL void few_rows_of(const bf16_t* __restrict__ x, const bf16_t* __restrict__ we, const int* __restrict__ token,
                        bf16_t* __restrict__ y, const GroupArgs& a, int r0, int hi, int turn, bf16_t* buf) {
  typedef FewTile<BN, BM> Sh;
  constexpr bool TWO = has_gate(KIND), OWN = of_own_row(KIND);
  constexpr int PER = TWO ? BN / 2 : BN;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, sub = lane >> 3;
  const int f0 = blockIdx.x * PER;
  const bf16_t *wsrc[Sh::WL], *xsrc[Sh::XL];
#pragma unroll
  for (int i = 0; i < Sh::XL; ++i) {
    const int r = BM >= 32 ? (wave * Sh::XL + i) * 8 + sub : wave * 4 + (sub & 3), at = min(r0 + r, hi - 1);
    xsrc[i] = x + (size_t)(OWN ? at : token[at]) * a.xs + ((lane & 7) ^ (r & 7)) * 8;
  }
#pragma unroll
  for (int i = 0; i < Sh::WL; ++i) {  // TWO: 8 gate rows and the same 8 up rows in turn
    const int r = (wave * Sh::WL + i) * 8 + sub;
    const size_t f = TWO ? min(f0 + (r >> 4) * 8 + (r & 7), a.F - 1) + ((r >> 3) & 1 ? (size_t)a.F : 0) : min(f0 + r, a.F - 1);
    wsrc[i] = we + f * a.kp + ((lane & 7) ^ (r & 7)) * 8;
  }
  floatx4 acc[Sh::R][Sh::C];
  stream_walk<Sh>(acc, buf, wsrc, xsrc, a.K / 64, turn, wave, lane);
  const int col = lane & 15, quad = lane >> 4;
#pragma unroll
  for (int j = 0; j < Sh::C; ++j) {
    const int row = r0 + Sh::wx(wave) + j * 16 + col;
#pragma unroll
    for (int i = 0; i < Sh::R; ++i) {
      const int w0 = Sh::wr(wave) + i * 16, f = f0 + (TWO ? w0 / 2 : w0) + quad * 4;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // lanes of quads 0 and 1 hold gates, those of 2 and 3 the products of up
        if (TWO) v[r] = siluf(acc[i][j][r]) * __shfl_xor(acc[i][j][r], 32);
        else v[r] = acc[i][j][r];
      }
      if (row < hi && f < a.F && (!TWO || quad < 2)) st4(y + (size_t)row * a.ys + f, v);  // F % 16 == 0
    }
  }
}
template <int KIND, int BN>
__global__ __launch_bounds__(256) void expert_few_kernel(const bf16_t* __restrict__ x, Listed w, const int* __restrict__ first,
                                                         const int* __restrict__ token, const int2* __restrict__ tiles,
                                                         bf16_t* __restrict__ y, bool turned, GroupArgs a) {
  extern __shared__ __attribute__((aligned(16))) bf16_t buf[];
  const int2 tile = tiles[blockIdx.y];
  const int e = __builtin_amdgcn_readfirstlane(tile.x);
  if (e < 0) return;
  int r0 = __builtin_amdgcn_readfirstlane(tile.y);
  const int hi = min(__builtin_amdgcn_readfirstlane(first[e + 1]), r0 + 128);
  const bf16_t* we = w.of(e, 0);
  // where rows lie a multiple of 4 KB apart blocks begin at different places of k (first_step of tile_ops.hip);
  // an expert's weights begin where all others' do
  const unsigned group = blockIdx.x * BN / 128 + e * 40503u, steps = a.K / 64;
  const int turn = turned ? (int)(((group * 2654435761u >> 16) * steps) >> 16) : 0;
  for (bool again = false; r0 < hi; again = true) {
    if (again) __syncthreads();  // LDS is read no more
    const int left = hi - r0;
    auto go = [&](auto most) {
      constexpr int BM = decltype(most)::value;
      few_rows_of<KIND, BN, BM>(x, we, token, y, a, r0, hi, turn, buf);
      r0 += BM;
    };
    if (left > 32) go(std::integral_constant<int, 64>());
    else if (left > 16) go(std::integral_constant<int, 32>());
    else go(std::integral_constant<int, 16>());
  }
}

// ---------------------------------------------------------------------------
// residual sum and norm
// ---------------------------------------------------------------------------

// x += mult * y (top 0) or mult * sum_j weight_j y[row_j]; h = norm(x; w_next).
// One block per token; the row stays in registers.
template <typename T, int V, int NC>
__global__ __launch_bounds__(256) void add_norm_kernel(
    const T* __restrict__ y, const int* __restrict__ rows, const float* __restrict__ weight, int top, int ys,
    float* __restrict__ x, const T* __restrict__ w_next, T* __restrict__ h, int D, float mult, float eps) {
  const size_t off = (size_t)blockIdx.x * D;
  __shared__ float red[4];
  float xv[NC * V], acc = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = (c * 256 + threadIdx.x) * V;
    float sum[V];
#pragma unroll
    for (int j = 0; j < V; ++j) xv[c * V + j] = sum[j] = 0.f;
    if (i < D) {
      ldv<V>(x + off + i, xv + c * V);
      if (top == 0) ldv<V>(y + (size_t)blockIdx.x * ys + i, sum);
      for (int k = 0; k < top; ++k) {
        const float wk = weight ? weight[(size_t)blockIdx.x * top + k] : 1.f;
        float v[V];
        ldv<V>(y + (size_t)rows[(size_t)blockIdx.x * top + k] * ys + i, v);
#pragma unroll
        for (int j = 0; j < V; ++j) sum[j] += wk * v[j];
      }
#pragma unroll
      for (int j = 0; j < V; ++j) {
        xv[c * V + j] += mult * sum[j];
        acc += xv[c * V + j] * xv[c * V + j];
      }
      stv<V>(x + off + i, xv + c * V);
    }
  }
  if (!w_next) return;
  const float inv = 1.f / sqrtf(block_sum(acc, red) / (float)D + eps);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = (c * 256 + threadIdx.x) * V;
    if (i < D) {
      float w[V], o[V];
      ldv<V>(w_next + i, w);
#pragma unroll
      for (int j = 0; j < V; ++j) o[j] = xv[c * V + j] * inv * (1.f + w[j]);
      stv<V>(h + off + i, o);
    }
  }
}

// ===========================================================================
// host side
// ===========================================================================

// x [.., D] -> (weights [T, top] fp32, row of every pair [T, top], token of
// every row, first row of every expert [E + 1], tiles [max + 1, 2], rows of a tile).
// `shared` experts follow the routed ones in every token's list (top counts
// them then); their weight is the sigmoid of one more row of w (gate) or one.
// on_input: the weights by row [T * top].
// w: the router's weights, or none: x are logits [T, E] that a router's own call has made
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, int64_t> route(Tensor x, OptT w, OptT correction, int64_t pick,
                                                                  int64_t groups, int64_t keep, double scale,
                                                                  bool softmax, int64_t shared, bool gate,
                                                                  bool on_input, int64_t tile_of, bool narrow) {
  const auto dt = io_type(x);
  const bool given = !w;
  CHK(!given || (shared == 0 && !narrow));
  if (!given) check_io(*w, dt);
  gate = gate && shared > 0;
  const int D = x.size(-1), T_ = x.numel() / D, E = given ? D : w->size(0) - gate;
  if (correction) { check_io(*correction, dt); CHK(correction->numel() == E); }
  CHK((given || (w->dim() == 2 && w->size(1) == D)) && T_ > 0 && shared >= 0);
  const int64_t top = pick + shared, all = E + shared;
  TORCH_CHECK(E >= 1 && all <= MAX_EXPERTS && pick >= 1 && pick <= MAX_PICK && pick <= E, "routing to ", pick, " of ", E,
              " experts and ", shared, " shared ones");
  TORCH_CHECK(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups && pick <= keep * (E / groups),
              "routing to ", pick, " experts of ", keep, " of ", groups, " groups of ", E, " experts");
  CHK((int64_t)T_ * top < INT_MAX);
  const int nblk = (T_ + RT - 1) / RT, pairs = T_ * (int)top;
  CHK(tile_of == 0 || tile_of == 128 || tile_of == 256);
  const int tile = tile_of ? (int)tile_of : pairs >= 320 * all ? 256 : 128, max_tiles = pairs / tile + std::min(pairs, (int)all);
  const auto ints = x.options().dtype(torch::kInt32);
  auto weight = f32(x, {T_, top});
  Tensor by_row;
  if (on_input) by_row = f32(x, {pairs});
  auto idx = torch::empty({T_, top}, ints), rank = torch::empty({T_, top}, ints), row = torch::empty({T_, top}, ints);
  auto counts = torch::empty({all, nblk}, ints), total = torch::empty({all}, ints), first = torch::empty({all + 1}, ints);
  auto token = torch::empty({pairs}, ints), tiles = torch::empty({max_tiles + 1, 2}, ints);
  const RouteArgs a{T_, D, E, (int)top, (int)groups, (int)keep, nblk, tile, (float)scale, (int)pick, (int)all, softmax, gate, narrow, given};
  const hipStream_t stream = cur_stream();
  CHK(groups <= 4 * 65);
  BY_TYPE(dt, {
    const T* cp = correction ? P<T>(*correction) : nullptr;
    auto run = [&](auto kernel, int waves) {
      const hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      TORCH_CHECK(err == hipSuccess, "no LDS for the router");
      const size_t lds = (2 * RT * E + waves * RT * 65) * sizeof(float) + RT * (top + 1) * sizeof(int);  // parts of 16 bytes
      hipLaunchKernelGGL(kernel, dim3(nblk), dim3(64 * waves), lds, stream, P<T>(x), given ? nullptr : P<T>(*w), cp,
                         idx.data_ptr<int>(), M<float>(weight), rank.data_ptr<int>(), counts.data_ptr<int>(), a);
    };
    // few tokens: more waves on each
    const bool few = nblk <= 256;
    if (!given && D % Frag<T>::K) run(route_kernel<T, false, MAX_EXPERTS / 16, 4>, 4);
    else if (E <= 64) { if (few) run(route_kernel<T, true, 4, 16>, 16); else run(route_kernel<T, true, 4, 4>, 4); }
    else if (E <= 256) { if (few) run(route_kernel<T, true, 16, 16>, 16); else run(route_kernel<T, true, 16, 4>, 4); }
    else run(route_kernel<T, true, MAX_EXPERTS / 16, 4>, 4);
  });
  if (nblk > FEW_BLOCKS)
    hipLaunchKernelGGL(count_scan_kernel, dim3(all), dim3(256), 0, stream, counts.data_ptr<int>(), total.data_ptr<int>(), nblk);
  hipLaunchKernelGGL(place_kernel, dim3((pairs + 255) / 256), dim3(256), 0, stream, idx.data_ptr<int>(),
                     rank.data_ptr<int>(), counts.data_ptr<int>(), total.data_ptr<int>(), P<float>(weight),
                     row.data_ptr<int>(), token.data_ptr<int>(), on_input ? M<float>(by_row) : nullptr,
                     first.data_ptr<int>(), (int2*)tiles.data_ptr<int>(), max_tiles, a);
  return {on_input ? by_row : weight, row, token, first, tiles, tile};
}

template <typename W>
static void launch_tiles(const W& w, const Tensor& x, const Tensor& token, const Tensor& first, const Tensor& tiles,
                         int64_t tile, int64_t kind, const GroupArgs& a, const Act& act, const float* by_row, Tensor& y) {
  const int max_tiles = tiles.size(0) - 1, pairs = token.numel(), rows = has_gate((int)kind) ? 2 * a.F : a.F;
  CHK(max_tiles >= 1);
  CHK(tile == 128 || tile == 256);
  // as many tiles as an expert has on average share its weight rows in a die's L2. us of the
  // gated product above, 3 and 4 of them: 2100 tokens (525 rows an expert) 903, 934; 4000
  // tokens (1000 rows) 1590, 1504
  const int group = pairs / (a.E * (int)tile) + 1;
  // few rows an expert: blocks of 128 weight rows, two to a CU, keep more of them on their
  // way: 25 and 50 rows 491 and 509 us (553 and 570 with 256); from 75 on 609 (589). So do those
  // that make one round of the chip: down of 8 experts of 4096 x 14336, 75 and 88 rows each, 200
  // and 203 us (220 and 226), but 280 (230) where uneven experts make more tiles than there are
  // CUs. From 88 rows on average on one expert in eight is taken to have a tile more, from 112 on one
  // in two. Experts of all sizes: 1.25 to 1.45 times as fast where that leaves half of the chip idle,
  // 1.1 to 1.2 up to the whole of it.
  const int64_t likely = pairs <= 88 * (int64_t)a.E ? std::min(pairs, a.E) : pairs <= 112 * (int64_t)a.E ? a.E + a.E / 8 : pairs / 128 + 1 + a.E / 2;
  const bool half = tile == 128 && (pairs <= 56 * (int64_t)a.E || likely * ((rows + 127) / 128) <= 256);
  const int bn = half ? 128 : 256, nf = (rows + bn - 1) / bn;
  // blocks that leave much of the chip idle, at 256 rows a tile, are planned by the kernel, which may
  // make tiles of 128 rows of them. The plan takes 1 to 4 us, and its grid is wider; the longer the
  // rows, the more blocks it is good for. Time with the router's tiles over time with the plan, on
  // average: up to 64 blocks 1.22 to 1.3 (K < 512: 1.09); to 128 0.88 (K < 512), 0.96 (< 1024), 1.0 (<
  // 2048), 1.05 (longer); to 256 0.85, 0.94, 0.99, 1.02 (< 4096), 1.05; to 384 0.86, 0.91, 0.96, 0.98, 1.0
  // (from 8192 on 1.01); to 512 0.99 at best
  const bool replan = tile == 256 && (int64_t)std::max(a.E, pairs / 256 + 1) * nf <= std::max(64, std::min(a.kp / 16, 384));
  const int most_tiles = replan ? pairs / 128 + std::min(pairs, a.E) : max_tiles;
  const dim3 grid(((most_tiles * nf + 7) / 8 + (tile == 256 ? DIE_CUS / 2 : 0)) * 8);
  auto run = [&](auto kernel, int lds) {
    const hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    TORCH_CHECK(err == hipSuccess, "no LDS for expert tiles");
    hipLaunchKernelGGL(kernel, grid, dim3(256), lds, cur_stream(), P<bf16_t>(x), w, first.data_ptr<int>(),
                       token.data_ptr<int>(), (const int2*)tiles.data_ptr<int>(), by_row, M<bf16_t>(y), max_tiles, group, 0, replan, a, act);
  };
  // where x takes 4 GB, offsets of gathered rows need more than 32 bits
  const bool far = !of_own_row((int)kind) && (uint64_t)x.numel() * 2 >= 0xffffffffull;
#define TILES(KIND, BN, TOK)                                                                                \
  {                                                                                                         \
    if (far) run(expert_tile_kernel<KIND, BN, TOK, !of_own_row(KIND), W>, expert_lds<BN, TOK>());            \
    else run(expert_tile_kernel<KIND, BN, TOK, false, W>, expert_lds<BN, TOK>());                            \
  }
#define TILES_OF(KIND) if (half) TILES(KIND, 128, 128) else if (tile == 256) TILES(KIND, 256, 256) else TILES(KIND, 256, 128)
  if constexpr (std::is_same<W, Listed>::value) {
    if (kind == SWIGLU) { TILES_OF(SWIGLU); }
    else { TILES_OF(PLAIN); }
  } else {
    if (kind == GATED) { TILES_OF(GATED); }
    else if (kind == RELU2) { TILES_OF(RELU2); }
    else { TILES_OF(PLAIN); }
  }
#undef TILES_OF
#undef TILES
}

// What the forms with one weight tensor per expert, bf16, take: SWIGLU ([2 F, K], gate rows
// first; x by token) or PLAIN ([F, K]; x by row), K % 64 == 0
static GroupArgs listed(Listed& list, const Tensor& x, const std::vector<Tensor>& w, const Tensor& token, const Tensor& first,
                        const Tensor& tiles, bool swiglu) {
  check_io(x, torch::kBFloat16);
  const int64_t E = w.size();
  CHK(x.dim() == 2 && E >= 1 && E <= MOST_LISTED && ((size_t)x.data_ptr() & 15) == 0);
  for (const Tensor& t : {token, first, tiles}) check_io(t, torch::kInt32);
  const int K = x.size(1), F_ = w[0].size(0) / (swiglu ? 2 : 1);
  CHK(first.numel() == E + 1 && K % 64 == 0 && F_ % 16 == 0 && (swiglu || x.size(0) == token.numel()));
  for (int64_t e = 0; e < E; ++e) {
    check_io(w[e], torch::kBFloat16);
    CHK(w[e].dim() == 2 && w[e].size(0) == F_ * (swiglu ? 2 : 1) && w[e].size(1) == K && ((size_t)w[e].data_ptr() & 15) == 0);
    list.w[e] = P<bf16_t>(w[e]);
  }
  return GroupArgs{K, K, F_, (int)E, K, F_};
}

// These by tiles.
Tensor expert_product_of(Tensor x, std::vector<Tensor> w, Tensor token, Tensor first, Tensor tiles, int64_t tile, bool swiglu) {
  Listed list{};
  const GroupArgs a = listed(list, x, w, token, first, tiles, swiglu);
  const int K = a.K, F_ = a.F, pairs = token.numel();
  const int64_t E = a.E;
  auto y = torch::empty({pairs, F_}, x.options());
  if (K <= 1 << 22) {
    launch_tiles(list, x, token, first, tiles, tile, swiglu ? SWIGLU : PLAIN, a, Act{}, nullptr, y);
    return y;
  }
  // offsets of a tile's weights have 32 bits: longer rows expert by expert, without tiles
  CHK(tile == 128 || tile == 256);
  auto stream = [&](auto kernel) {
    for (int64_t e = 0; e < E; ++e)
      hipLaunchKernelGGL(kernel, dim3(F_ / 16), dim3(256), 0, cur_stream(), P<bf16_t>(x), list.w[e], first.data_ptr<int>() + e,
                         token.data_ptr<int>(), (const float*)nullptr, M<bf16_t>(y), a, Act{});
  };
  if (swiglu) stream(expert_stream_kernel<bf16_t, SWIGLU, true>);
  else stream(expert_stream_kernel<bf16_t, PLAIN, true>);
  return y;
}

// The same of few tokens, tiles of 128 rows
Tensor expert_few_of(Tensor x, std::vector<Tensor> w, Tensor token, Tensor first, Tensor tiles, int64_t tile, bool swiglu) {
  CHK(tile == 128 && tiles.dim() == 2 && tiles.size(0) >= 2 && tiles.size(0) <= 65536);
  Listed list{};
  const GroupArgs a = listed(list, x, w, token, first, tiles, swiglu);
  const int pairs = token.numel();
  auto y = torch::empty({pairs, a.F}, x.options());
  const bool turned = a.K <= 16384 && a.K % 2048 == 0;
  auto run = [&](auto kernel, int lds, int per) {
    const hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    TORCH_CHECK(err == hipSuccess, "no LDS for experts of few rows");
    hipLaunchKernelGGL(kernel, dim3((a.F + per - 1) / per, (unsigned)tiles.size(0) - 1), dim3(256), lds, cur_stream(), P<bf16_t>(x), list,
                       first.data_ptr<int>(), token.data_ptr<int>(), (const int2*)tiles.data_ptr<int>(), M<bf16_t>(y), turned, a);
  };
  // 128 weight rows a block from 16 rows an expert on, so that rows are read half as often: us with 64 and so,
  // the experts above: 64 tokens 450, 445; 128 491, 460; 192 568, 467; 32 tokens 440, 441; the smaller ones
  // 32 tokens 202, 208; 128 230, 232
  if (pairs >= 16 * a.E) {
    if (swiglu) run(expert_few_kernel<SWIGLU, 128>, few_lds<128>(), 64);
    else run(expert_few_kernel<PLAIN, 128>, few_lds<128>(), 128);
  } else {
    if (swiglu) run(expert_few_kernel<SWIGLU, 64>, few_lds<64>(), 32);
    else run(expert_few_kernel<PLAIN, 64>, few_lds<64>(), 64);
  }
  return y;
}

// One grouped product over all pairs: GATED (x by token, weights [E,2,F,kp]),
// RELU2 (x by token, weights [E,F,kp]) or PLAIN (x by row, weights [E,F,kp]); kp:
// row length padded with zeros. by_row [pairs]: scales of the product's rows.
Tensor expert_product(Tensor x, Tensor w, Tensor token, Tensor first, Tensor tiles, int64_t tile, int64_t kind,
                      double alpha, double limit, double plus, OptT by_row) {
  const auto dt = io_type(x);
  check_io(w, dt);
  CHK(kind == PLAIN || kind == GATED || kind == RELU2);
  const bool gated_ = kind == GATED;
  CHK(w.dim() == (gated_ ? 4 : 3) && x.dim() == 2);
  for (const Tensor& t : {token, first, tiles}) check_io(t, torch::kInt32);
  const int E = w.size(0), F_ = w.size(-2), kp = w.size(-1), K = x.size(1), pairs = token.numel();
  CHK((!gated_ || w.size(1) == 2) && first.numel() == E + 1 && K <= kp && kp % 64 == 0 && F_ % 16 == 0 && kp - K < 64);
  CHK(kind != PLAIN || x.size(0) == pairs);
  if (by_row) { check_io(*by_row, torch::kFloat32); CHK(kind != PLAIN && by_row->numel() == pairs); }
  const float* bp = by_row ? P<float>(*by_row) : nullptr;
  auto y = torch::empty({pairs, F_}, x.options());
  const GroupArgs a{K, kp, F_, E, K, F_};
  const Act act{(float)alpha, (float)limit, (float)plus};
  const hipStream_t stream = cur_stream();
  const int *fp = first.data_ptr<int>(), *tp = token.data_ptr<int>();
  // on average more than 24 rows per expert: weights are worth tiling
  if (dt == torch::kBFloat16 && K % 8 == 0 && kp <= 1 << 22 && pairs > 24 * E) {
    launch_tiles(Stacked{P<bf16_t>(w)}, x, token, first, tiles, tile, kind, a, act, bp, y);
    return y;
  }
  const dim3 grid(F_ / 16, E);
#define STREAM(KIND, WHOLE)                                                                                     \
  hipLaunchKernelGGL((expert_stream_kernel<T, KIND, WHOLE>), grid, dim3(256), 0, stream, P<T>(x), P<T>(w), fp,     \
                     tp, bp, M<T>(y), a, act)
#define STREAM_OF(KIND) if (K % Frag<T>::K == 0) STREAM(KIND, true); else STREAM(KIND, false);
  BY_TYPE(dt, {
    if (kind == GATED) { STREAM_OF(GATED) }
    else if (kind == RELU2) { STREAM_OF(RELU2) }
    else { STREAM_OF(PLAIN) }
  });
#undef STREAM_OF
#undef STREAM
  return y;
}

// x += mult * y, or mult * the weighted rows of y; returns the stream's norm
OptT add_norm(Tensor y, OptT rows, OptT weight, Tensor x, OptT w_next, double mult, double eps) {
  const auto dt = io_type(y);
  check_io(x, torch::kFloat32);
  const int D = x.size(-1), n = x.numel() / D, ys = y.size(-1);
  int top = 0;
  if (rows) {
    check_io(*rows, torch::kInt32);
    if (weight) { check_io(*weight, torch::kFloat32); CHK(weight->numel() == rows->numel()); }
    top = rows->size(-1);
    CHK(rows->numel() == (int64_t)n * top && y.numel() == (int64_t)n * top * ys && ys >= D);
  } else {
    CHK(y.numel() == x.numel() && ys == D);
  }
  OptT h;
  if (w_next) { check_io(*w_next, dt); CHK(w_next->numel() == D); h = torch::empty(x.sizes(), x.options().dtype(dt)); }
  if (n == 0) return h;
  const int* rp = rows ? rows->data_ptr<int>() : nullptr;
  const float* wp = weight ? weight->data_ptr<float>() : nullptr;
#define NORM(V, NC)                                                                                            \
  if (nc <= NC) {                                                                                              \
    hipLaunchKernelGGL((add_norm_kernel<T, V, NC>), dim3(n), dim3(256), 0, cur_stream(), P<T>(y), rp, wp, top, ys, \
                       M<float>(x), wn, hp, D, (float)mult, (float)eps);                                       \
    return h;                                                                                                  \
  }
  BY_TYPE(dt, {
    const T* wn = w_next ? P<T>(*w_next) : nullptr;
    T* hp = h ? M<T>(*h) : nullptr;
    if (D % 4 == 0 && ys % 4 == 0) {
      const int nc = (D + 1023) / 1024;
      NORM(4, 1) NORM(4, 2) NORM(4, 4) NORM(4, 8) NORM(4, 16)
    } else {
      const int nc = (D + 255) / 256;
      NORM(1, 1) NORM(1, 4) NORM(1, 16)
    }
  });
#undef NORM
  TORCH_CHECK(false, "row of ", D, " elements is too long");
}

// silu of gate and up of all rows of x, bf16: w [2 F, K], gate rows first; K % 64 == 0. The
// product bounds it; a library's product, with the activation's kernel behind it that reads
// and writes what this one never stores, took, us: 320 tokens by [16384, 2048] 29 (24 so);
// 700 by [28672, 4096] 160 (145); 3000 by [37888, 3584] 728 (591); 8192 by [17920, 1536] 452
// (358). Whole rounds of large tiles are all a library needs: 8192 by [57344, 8192] 5168 (5390).
Tensor gate_product(Tensor x, Tensor w) {
  check_io(x, torch::kBFloat16);
  check_io(w, torch::kBFloat16);
  CHK(x.dim() == 2 && w.dim() == 2 && (((size_t)x.data_ptr() | (size_t)w.data_ptr()) & 15) == 0);
  const int64_t rows = x.size(0), K = x.size(1), F_ = w.size(0) / 2;
  CHK(rows >= 1 && rows <= 1 << 22 && K >= 64 && K <= 1 << 22 && K % 64 == 0 && w.size(1) == K);
  CHK(w.size(0) >= 32 && w.size(0) <= 1 << 22 && w.size(0) % 32 == 0);
  auto y = torch::empty({rows, F_}, x.options());
  // tiles of up to 256 rows, or, up to some ten rounds, of fewer where the rounds they make take
  // less time by what plan_of goes by. us, least tiles first: 600 and 700 rows by [16384, 2048] 45.6
  // and 49.4, 39.4 and 44.6; 512 by [17920, 1536] 37.2, 32.0; 300 and 1000 by [9728, 896] 13.1 and
  // 24.0, 10.3 and 21.3; larger weights the same
  const int nf = (int)((F_ + 127) / 128), least = (int)((rows + 255) / 256);
  auto share_of = [&](int n) { return ((rows + n - 1) / n + 31) / 32 * 32; };
  auto time = [&](int n) {
    const int64_t all = ((int64_t)n * nf + 7) / 8, left = all % DIE_CUS;  // of a die
    return ((double)(all / DIE_CUS) + (left == 0 ? 0 : left <= DIE_CUS / 2 ? 0.62 : 1)) * (0.4 + 0.00375 * std::max<int64_t>(128, share_of(n)));
  };
  int tiles = least;
  if ((int64_t)least * nf < 2560)
    for (int n = least + 1; n <= 2 * least; ++n) {
      const int some = (int)((rows + share_of(n) - 1) / share_of(n));  // none without a row
      if (time(some) < 0.95 * time(least) && time(some) < time(tiles)) tiles = some;
    }
  // panels of 2, 4, 6 and 8 tiles, us: 1500 rows of 3584 by 37888 326, 320, 315, 312; 6001 by
  // [28672, 4096] 1047, 1030, 1005, 1022; 3000 by [57344, 8192] 2114, 2058, 1988, 2022
  const int group = 6;
  auto kernel = expert_tile_kernel<DENSE, 256, 256, false, Stacked>;
  constexpr int lds = expert_lds<256, 256>();
  const hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  TORCH_CHECK(err == hipSuccess, "no LDS for gate and up");
  hipLaunchKernelGGL(kernel, dim3(((tiles * nf + 7) / 8 + DIE_CUS / 2) * 8), dim3(256), lds, cur_stream(), P<bf16_t>(x),
                     Stacked{P<bf16_t>(w)}, (const int*)nullptr, (const int*)nullptr, (const int2*)nullptr, (const float*)nullptr,
                     M<bf16_t>(y), tiles, group, (int)rows, false, GroupArgs{(int)K, (int)K, (int)F_, 1, (int)K, (int)F_}, Act{});
  return y;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("route", &route, "router: sigmoid scores or a softmax over the chosen, group-limited top-k, shared experts; rows of all pairs",
        py::arg("x"), py::arg("w"), py::arg("correction"), py::arg("top"), py::arg("groups"), py::arg("keep"),
        py::arg("scale"), py::arg("softmax") = false, py::arg("shared") = 0, py::arg("gate") = true,
        py::arg("on_input") = false, py::arg("tile") = 0, py::arg("narrow") = false);
  m.def("expert_product", &expert_product, "grouped product of all (token, expert) pairs, with an activation or plain",
        py::arg("x"), py::arg("w"), py::arg("token"), py::arg("first"), py::arg("tiles"), py::arg("tile"), py::arg("kind"),
        py::arg("alpha") = 0.0, py::arg("limit") = 0.0, py::arg("plus") = 0.0, py::arg("by_row") = py::none());
  m.def("expert_product_of", &expert_product_of, "the same by tiles, with one weight tensor per expert: silu of gate and up, or plain");
  m.def("readable", [](const Tensor& x, const std::vector<Tensor>& w) {
    for (const Tensor& t : w)
      if (!t.is_cuda() || t.device() != x.device() || t.scalar_type() != torch::kBFloat16 || !t.is_contiguous() || ((size_t)t.data_ptr() & 15))
        return false;
    return ((size_t)x.data_ptr() & 15) == 0;
  }, "whether grouped products of x may read these weights: bf16 on its device, contiguous, on 16 bytes");
  m.def("expert_few_of", &expert_few_of, "the same of few tokens");
  m.attr("PLAIN") = (int)PLAIN;
  m.attr("GATED") = (int)GATED;
  m.attr("RELU2") = (int)RELU2;
  m.def("gate_product", &gate_product, "silu of gate and up of all rows, by the same tiles");
  m.def("add_norm", &add_norm, "stream += mult * (output or weighted expert rows); norm of the stream");
}
