// Causal GQA attention of a training pass and its gradients, from the fused projection
// to the heads' outputs (head dim 64 or 128; the reference trains through torch's
// attention, general_mha.py:211-226).
//
// Queries, keys and values are bf16, and so are the outputs' gradients: their products
// are exact on the bf16 matrix cores and summed in fp32. Probabilities and the
// gradients of scores stay fp32: they enter products as three bf16 parts each, which
// hold all 24 bits. What bounds these kernels are the matrix cores (4 products forward,
// 13 backward for every pair of a query and a key) and the splitting; scores are
// computed again rather than stored, twice backward, so that every gradient is summed
// in one place and in order.
//
// Tensors lie in fragment order, once by rows and once transposed, as the packed cache
// does: every load of a wave is 1 KB in one piece, and no kernel needs LDS for a
// product. Scores are computed from rows in an order in which the lane that holds a
// column's numbers feeds them to the next product. What is left to hide are the loads:
// the next tile's are on their way while one is worked on (without: 88 us forward, 197
// and 72 backward, below).
// 8 x 512 tokens, 32 heads of 128 on 8: 62 us forward, 116 for keys and values, 64 for
// queries, 62 packing (150 and 170 MB); torch's fp32 attention with its copies: 487 us
// forward and 1550 backward. 4 x 512, 32 heads of 64 on 4: 25, 48, 24 and 17; 143 and
// 398. Errors against 64 bits are below torch's fp32 attention's (1.2e-7 for 1.7e-7).
#include "common.h"

struct TrainArgs {
  const bf16_t *qkv, *dout;
  bf16_t *r, *t;            // packed qkv by rows and transposed: [B][H + 2 KVH][S32 * HD]
  bf16_t *dr, *dt;          // the same of the outputs' gradients: [B][H][S32 * HD]
  bf16_t *out, *dqkv;
  float *o, *lse, *delta;   // fp32 [B, S, H HD]; [B][H][S32], lse to base 2
  const float *cos, *sin;
  const int* positions;
  int B, S, S32, H, KVH, per_row, places;  // places: rows of the rotation's tables
  float scale;
};

// where a token stands in the tables
DEVINL int place(const TrainArgs& a, int b, int s) {
  return table_row(a.positions[a.per_row ? b * a.S + s : s], a.places);
}

// The 32 rows of one head from tile s0 on, in LDS, to both orders
template <int HD>
DEVINL void pack_tile(const bf16_t (*tile)[HD + 8], bf16_t* r, bf16_t* t, int s0, int S32) {
  constexpr int KC = HD / 32, VG = HD / 16;
  for (int i = threadIdx.x; i < 2 * KC * 64; i += 256) {
    const int lane = i & 63, c = i / 64 % KC, half = i / 64 / KC;
    *(bf16x8*)(r + (((size_t)(s0 / 16 + half) * KC + c) * 64 + lane) * 8) =
        *(const bf16x8*)(&tile[half * 16 + (lane & 15)][c * 32 + (lane >> 4) * 8]);
  }
  for (int i = threadIdx.x; i < VG * 64; i += 256) {
    const int lane = i & 63, g = i / 64;
    union { bf16x8 v; bf16_t e[8]; } u;
#pragma unroll
    for (int j = 0; j < 8; ++j) u.e[j] = tile[(lane >> 4) * 8 + j][g * 16 + (lane & 15)];
    *(bf16x8*)(t + (((size_t)g * (S32 / 32) + s0 / 32) * 64 + lane) * 8) = u.v;
  }
}

// A block packs 32 tokens of one slot (a query, key or value head), rotated. Rows past
// the last token are zeros.
template <int HD>
__global__ __launch_bounds__(256) void pack_qkv_kernel(TrainArgs a) {
  __shared__ __attribute__((aligned(16))) bf16_t tile[32][HD + 8];
  const int slots = a.H + 2 * a.KVH, slot = blockIdx.y, b = blockIdx.z, s0 = blockIdx.x * 32;
  for (int i = threadIdx.x; i < 32 * (HD / 8); i += 256) {
    const int c = i % (HD / 8) * 4, row = i / (HD / 8), s = s0 + row;
    float x1[4] = {}, x2[4] = {};
    if (s < a.S) {
      const bf16_t* src = a.qkv + (((size_t)b * a.S + s) * slots + slot) * HD + c;
      ld4(src, x1);
      ld4(src + HD / 2, x2);
      if (slot < a.H + a.KVH) {
        float co[4], si[4];
        const int pos = place(a, b, s);
        ld_angles(a.cos, pos, HD / 2, c, co);
        ld_angles(a.sin, pos, HD / 2, c, si);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float y1 = x1[j] * co[j] - x2[j] * si[j], y2 = x2[j] * co[j] + x1[j] * si[j];
          x1[j] = y1;
          x2[j] = y2;
        }
      }
    }
    st4(&tile[row][c], x1);
    st4(&tile[row][c + HD / 2], x2);
  }
  __syncthreads();
  const size_t at = ((size_t)b * slots + slot) * a.S32 * HD;
  pack_tile<HD>(tile, a.r + at, a.t + at, s0, a.S32);
}

// The same for 32 tokens of one head of the outputs' gradients, and delta = dout . o
template <int HD>
__global__ __launch_bounds__(256) void pack_dout_kernel(TrainArgs a) {
  __shared__ __attribute__((aligned(16))) bf16_t tile[32][HD + 8];
  const int h = blockIdx.y, b = blockIdx.z, s0 = blockIdx.x * 32;
  const int row = threadIdx.x >> 3, part = threadIdx.x & 7, s = s0 + row;  // 8 threads a token
  const size_t tok = (((size_t)b * a.S + s) * a.H + h) * HD;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < HD / 32; ++i) {
    const int c = (i * 8 + part) * 4;
    ushort4_t d = {0, 0, 0, 0};
    if (s < a.S) {
      d = *(const ushort4_t*)(a.dout + tok + c);
      float v[4], o[4];
      ld4(a.dout + tok + c, v);
      ld4(a.o + tok + c, o);
#pragma unroll
      for (int j = 0; j < 4; ++j) sum += v[j] * o[j];
    }
    *(ushort4_t*)&tile[row][c] = d;
  }
#pragma unroll
  for (int m = 1; m < 8; m <<= 1) sum += __shfl_xor(sum, m);
  if (part == 0) a.delta[((size_t)b * a.H + h) * a.S32 + s] = sum;
  __syncthreads();
  const size_t at = ((size_t)b * a.H + h) * a.S32 * HD;
  pack_tile<HD>(tile, a.dr + at, a.dt + at, s0, a.S32);
}

// Fragments of 16 rows in order, and of 32 rows in the order for the next product
// (row i of product hf is i / 4 * 8 + i % 4 + 4 hf)
template <int HD>
DEVINL void load_rows(const bf16_t* r, int tile16, int lane, bf16x8* f) {
#pragma unroll
  for (int c = 0; c < HD / 32; ++c) f[c] = *(const bf16x8*)(r + (((size_t)tile16 * (HD / 32) + c) * 64 + lane) * 8);
}
template <int HD>
DEVINL const bf16_t* mixed_base(const bf16_t* r, int lane) {
  const int p = ((lane & 15) >> 2) * 8 + (lane & 3);
  return r + ((size_t)(p >> 4) * (HD / 32) * 64 + (lane >> 4) * 16 + (p & 15)) * 8;
}
// all of the 32 rows of `tile` (by mixed_base)
template <int HD>
DEVINL void load_mixed(const bf16_t* mixed, int tile, bf16x8 (*m)[HD / 32]) {
#pragma unroll
  for (int hf = 0; hf < 2; ++hf)
#pragma unroll
    for (int c = 0; c < HD / 32; ++c) m[hf][c] = *(const bf16x8*)(mixed + (size_t)tile * (HD * 32) + c * 512 + hf * 32);
}
// the transposed fragments of the same 32 rows
template <int HD>
DEVINL void load_turned(const bf16_t* t, int tile, int tiles, bf16x8* m) {
#pragma unroll
  for (int g = 0; g < HD / 16; ++g) m[g] = *(const bf16x8*)(t + ((size_t)g * tiles + tile) * 512);
}
// their scores with N times 16 columns: a lane's column with rows quad * 8 + 0..7
template <int HD, int N>
DEVINL void scores(const bf16x8 (*m)[HD / 32], const bf16x8 (*f)[HD / 32], float (*v)[8]) {
  floatx4 s[N][2];
#pragma unroll
  for (int hf = 0; hf < 2; ++hf)
#pragma unroll
    for (int t = 0; t < N; ++t) {
      s[t][hf] = (floatx4)(0.f);
#pragma unroll
      for (int c = 0; c < HD / 32; ++c) s[t][hf] = mma(m[hf][c], f[t][c], s[t][hf]);
    }
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int i = 0; i < 8; ++i) v[t][i] = s[t][i >> 2][i & 3];
}
// loads before stay before, and what follows after
DEVINL void fence() { __builtin_amdgcn_sched_barrier(0); }

DEVINL float quad_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16));
  return fmaxf(v, __shfl_xor(v, 32));
}

// A wave has 32 queries of a head and walks the keys up to them.
template <int HD>
__global__ __launch_bounds__(256, 2) void train_forward_kernel(TrainArgs a) {
  constexpr int KC = HD / 32, VG = HD / 16, QT = 2;
  const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4, tiles = a.S32 / 32;
  const int wid = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (wid >= a.B * a.H * tiles) return;
  const int bh = wid % (a.B * a.H), tile = tiles - 1 - wid / (a.B * a.H), b = bh / a.H, h = bh % a.H;  // the longest first
  const int slots = a.H + 2 * a.KVH, kvh = h / (a.H / a.KVH);
  const size_t head = (size_t)a.S32 * HD;
  const bf16_t* q = a.r + ((size_t)b * slots + h) * head;
  const bf16_t* k = mixed_base<HD>(a.r + ((size_t)b * slots + a.H + kvh) * head, lane);
  const bf16_t* v = a.t + ((size_t)b * slots + a.H + a.KVH + kvh) * head + lane * 8;
  bf16x8 qf[QT][KC];
  float m[QT], l[QT];
  floatx4 o[QT][VG];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    load_rows<HD>(q, tile * 2 + t, lane, qf[t]);
    m[t] = -1e30f;
    l[t] = 0.f;
#pragma unroll
    for (int g = 0; g < VG; ++g) o[t][g] = (floatx4)(0.f);
  }
  const float scale = a.scale * 1.4426950408889634f;
  bf16x8 km[2][KC];
  load_mixed<HD>(k, 0, km);
  for (int j = 0; j <= tile; ++j) {
    bf16x8 pf[QT][3], vf[VG];
    float st[QT][8];
    load_turned<HD>(v, j, tiles, vf);
    fence();
    scores<HD, QT>(km, qf, st);
    fence();
    load_mixed<HD>(k, min(j + 1, tile), km);
    fence();
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      float* s = st[t];
      float top = m[t];
      const int d = j == tile ? t * 16 + col - quad * 8 : 8;  // keys past the query, in the last tile
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        s[i] = i <= d ? s[i] * scale : -INFINITY;
        top = fmaxf(top, s[i]);
      }
      if (__any(top > m[t])) {
        top = quad_max(top);
        const float f = __builtin_amdgcn_exp2f(m[t] - top);
        m[t] = top;
        l[t] *= f;
#pragma unroll
        for (int g = 0; g < VG; ++g) o[t][g] *= f;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        s[i] = __builtin_amdgcn_exp2f(s[i] - m[t]);
        l[t] += s[i];
      }
      split3(s, pf[t]);
    }
#pragma unroll
    for (int g = 0; g < VG; ++g)
#pragma unroll
      for (int t = 0; t < QT; ++t) o[t][g] = mma3(vf[g], pf[t], o[t][g]);
  }
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int s = tile * 32 + t * 16 + col;
    float sum = l[t] + __shfl_xor(l[t], 16);
    sum += __shfl_xor(sum, 32);
    // rows past the last token see only zeros: their probabilities must stay finite
    if (quad == 0) a.lse[(size_t)bh * a.S32 + s] = m[t] + __builtin_amdgcn_logf(sum);
    if (s >= a.S) continue;
    const float f = 1.f / sum;
    const size_t at = (((size_t)b * a.S + s) * a.H + h) * HD + quad * 4;
#pragma unroll
    for (int g = 0; g < VG; ++g) {
      o[t][g] *= f;
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = o[t][g][i];
      st4(a.o + at + g * 16, y);
      st4(a.out + at + g * 16, y);
    }
  }
}

// The rotation's transpose on a lane's column (channels g * 16 + quad * 4 + 0..3), each
// gradient rounded before and after, to bf16 rows
template <int HD>
DEVINL void turn_back(const TrainArgs& a, floatx4* o, int b, int s, int quad, bf16_t* dst, bool turn) {
  constexpr int VG = HD / 16;
  const int pos = turn ? place(a, b, s) : 0;
#pragma unroll
  for (int g = 0; g < VG / 2; ++g) {
    float y1[4], y2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y1[i] = o[g][i];
      y2[i] = o[g + VG / 2][i];
    }
    if (turn) {
      float co[4], si[4];
      ld_angles(a.cos, pos, HD / 2, g * 16 + quad * 4, co);
      ld_angles(a.sin, pos, HD / 2, g * 16 + quad * 4, si);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bf16_t r1 = f2b(y1[i]), r2 = f2b(y2[i]);
        const float g1 = ld(&r1), g2 = ld(&r2);
        y1[i] = g1 * co[i] + g2 * si[i];
        y2[i] = g2 * co[i] - g1 * si[i];
      }
    }
    st4(dst + g * 16 + quad * 4, y1);
    st4(dst + (g + VG / 2) * 16 + quad * 4, y2);
  }
}

// Queries' gradients: a wave has 32 queries of a head.
template <int HD>
__global__ __launch_bounds__(256, 2) void train_dq_kernel(TrainArgs a) {
  constexpr int KC = HD / 32, VG = HD / 16, QT = 2;
  const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4, tiles = a.S32 / 32;
  const int wid = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (wid >= a.B * a.H * tiles) return;
  const int bh = wid % (a.B * a.H), tile = tiles - 1 - wid / (a.B * a.H), b = bh / a.H, h = bh % a.H;
  const int slots = a.H + 2 * a.KVH, kvh = h / (a.H / a.KVH);
  const size_t head = (size_t)a.S32 * HD;
  const bf16_t* k = mixed_base<HD>(a.r + ((size_t)b * slots + a.H + kvh) * head, lane);
  const bf16_t* v = mixed_base<HD>(a.r + ((size_t)b * slots + a.H + a.KVH + kvh) * head, lane);
  const bf16_t* kt = a.t + ((size_t)b * slots + a.H + kvh) * head + lane * 8;
  bf16x8 qf[QT][KC], df[QT][KC];
  float lse[QT], delta[QT];
  floatx4 o[QT][VG];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    load_rows<HD>(a.r + ((size_t)b * slots + h) * head, tile * 2 + t, lane, qf[t]);
    load_rows<HD>(a.dr + (size_t)bh * head, tile * 2 + t, lane, df[t]);
    lse[t] = a.lse[(size_t)bh * a.S32 + tile * 32 + t * 16 + col];
    delta[t] = a.delta[(size_t)bh * a.S32 + tile * 32 + t * 16 + col];
#pragma unroll
    for (int g = 0; g < VG; ++g) o[t][g] = (floatx4)(0.f);
  }
  const float scale = a.scale * 1.4426950408889634f;
  bf16x8 km[2][KC];
  load_mixed<HD>(k, 0, km);
  for (int j = 0; j <= tile; ++j) {
    bf16x8 sf[QT][3], kf[VG], vm[2][KC];
    float st[QT][8], dpt[QT][8];
    load_mixed<HD>(v, j, vm);
    fence();
    scores<HD, QT>(km, qf, st);
    fence();
    load_mixed<HD>(k, min(j + 1, tile), km);
    fence();
    scores<HD, QT>(vm, df, dpt);
    fence();
    load_turned<HD>(kt, j, tiles, kf);
    fence();
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      float *s = st[t], *dp = dpt[t];
      const int d = j == tile ? t * 16 + col - quad * 8 : 8;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        s[i] = i <= d ? __builtin_amdgcn_exp2f(s[i] * scale - lse[t]) * (dp[i] - delta[t]) * a.scale : 0.f;
      split3(s, sf[t]);
    }
#pragma unroll
    for (int g = 0; g < VG; ++g)
#pragma unroll
      for (int t = 0; t < QT; ++t) o[t][g] = mma3(kf[g], sf[t], o[t][g]);
  }
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int s = tile * 32 + t * 16 + col;
    if (s < a.S) turn_back<HD>(a, o[t], b, s, quad, a.dqkv + (((size_t)b * a.S + s) * slots + h) * HD, true);
  }
}

// Keys' and values' gradients: KW waves of a block have KT * 16 positions of a key head
// each and walk the queries from them on, of all heads that share it, in step (what one
// loads, the others find in L1); G such groups share the walk and add up in LDS.
// Head dim 128: 2 x 16 positions halve the loads of a product, at one wave a SIMD with
// all registers (116 us, 128 with one wave to a walk, 213 with 16 positions a wave).
// 64: 16 positions and 8 waves a block fill the chip sooner (48 us, 54 with 2 x 16).
template <int HD, int KT, int KW, int G>
__global__ __launch_bounds__(KW * G * 64, 1) void train_dkv_kernel(TrainArgs a) {
  constexpr int KC = HD / 32, VG = HD / 16;
  __shared__ floatx4 red[G > 1 ? G / 2 * KW : 1][2 * VG][64];
  const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4, tiles = a.S32 / 32, rep = a.H / a.KVH;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = wave % KW, group = wave / KW;
  const int bh = blockIdx.x % (a.B * a.KVH), block = blockIdx.x / (a.B * a.KVH), b = bh / a.KVH, kvh = bh % a.KVH;
  const int tile16 = (block * KW + w) * KT, j0 = block * KW * KT / 2, nj = tiles - j0, slots = a.H + 2 * a.KVH;
  const size_t head = (size_t)a.S32 * HD;
  bf16x8 kf[KT][KC], vf[KT][KC];
  floatx4 dk[KT][VG], dv[KT][VG];
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const int at = min(tile16 + t, tiles * 2 - 1);
    load_rows<HD>(a.r + ((size_t)b * slots + a.H + kvh) * head, at, lane, kf[t]);
    load_rows<HD>(a.r + ((size_t)b * slots + a.H + a.KVH + kvh) * head, at, lane, vf[t]);
#pragma unroll
    for (int g = 0; g < VG; ++g) dk[t][g] = dv[t][g] = (floatx4)(0.f);
  }
  const float scale = a.scale * 1.4426950408889634f;
  const bf16_t* q = mixed_base<HD>(a.r + ((size_t)b * slots + kvh * rep) * head, lane);
  const bf16_t* d = mixed_base<HD>(a.dr + ((size_t)b * a.H + kvh * rep) * head, lane);
  const bf16_t* qt = a.t + ((size_t)b * slots + kvh * rep) * head + lane * 8;
  const bf16_t* dt = a.dt + ((size_t)b * a.H + kvh * rep) * head + lane * 8;
  const float* lse = a.lse + ((size_t)b * a.H + kvh * rep) * a.S32 + quad * 8;
  const float* delta = a.delta + ((size_t)b * a.H + kvh * rep) * a.S32 + quad * 8;
  bf16x8 qm[2][KC], dm[2][KC];
  int h = group / nj, j = j0 + group % nj;
  if (h < rep) {
    load_mixed<HD>(q + h * head, j, qm);
    load_mixed<HD>(d + h * head, j, dm);
  }
  while (h < rep) {
    float ls[8], de[8], s[KT][8], dp[KT][8];
    bf16x8 pf[KT][3], sf[KT][3], qf[VG], df[VG];
    const int here = j;
    ld4(lse + (size_t)h * a.S32 + j * 32, ls);
    ld4(lse + (size_t)h * a.S32 + j * 32 + 4, ls + 4);
    ld4(delta + (size_t)h * a.S32 + j * 32, de);
    ld4(delta + (size_t)h * a.S32 + j * 32 + 4, de + 4);
    load_turned<HD>(dt + h * head, j, tiles, df);
    load_turned<HD>(qt + h * head, j, tiles, qf);
    fence();
    scores<HD, KT>(qm, kf, s);
    scores<HD, KT>(dm, vf, dp);
    fence();
    for (j += G; j >= tiles; j -= nj) ++h;
    load_mixed<HD>(q + min(h, rep - 1) * head, j, qm);
    load_mixed<HD>(d + min(h, rep - 1) * head, j, dm);
    fence();
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const int first = (tile16 + t) * 16 + col - here * 32 - quad * 8;  // queries before the key don't see it
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float p = i >= first ? __builtin_amdgcn_exp2f(s[t][i] * scale - ls[i]) : 0.f;
        dp[t][i] = p * (dp[t][i] - de[i]) * a.scale;
        s[t][i] = p;
      }
      split3(s[t], pf[t]);
      split3(dp[t], sf[t]);
    }
#pragma unroll
    for (int g = 0; g < VG; ++g)
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        dv[t][g] = mma3(df[g], pf[t], dv[t][g]);
        dk[t][g] = mma3(qf[g], sf[t], dk[t][g]);
      }
  }
#pragma unroll
  for (int t = 0; t < KT; ++t) {
#pragma unroll
    for (int step = G / 2; step >= 1; step >>= 1) {
      if (group >= step && group < 2 * step)
#pragma unroll
        for (int g = 0; g < VG; ++g) {
          red[wave - step * KW][g][lane] = dk[t][g];
          red[wave - step * KW][VG + g][lane] = dv[t][g];
        }
      __syncthreads();
      if (group < step)
#pragma unroll
        for (int g = 0; g < VG; ++g) {
          dk[t][g] += red[wave][g][lane];
          dv[t][g] += red[wave][VG + g][lane];
        }
      __syncthreads();
    }
    const int pos = (tile16 + t) * 16 + col;
    if (group == 0 && pos < a.S) {
      bf16_t* dst = a.dqkv + (((size_t)b * a.S + pos) * slots + a.H + kvh) * HD;
      turn_back<HD>(a, dk[t], b, pos, quad, dst, true);
      turn_back<HD>(a, dv[t], b, pos, quad, dst + (size_t)a.KVH * HD, false);
    }
  }
}

// ===========================================================================
// host side
// ===========================================================================

static TrainArgs train_args(const Tensor& qkv, const Tensor& cos, const Tensor& sin, const Tensor& positions, int64_t H,
                            int64_t KVH, int64_t hd) {
  check_io(qkv, torch::kBFloat16);
  check_io(cos, torch::kFloat32);
  check_io(sin, torch::kFloat32);
  check_io(positions, torch::kInt32);
  CHK((hd == 64 || hd == 128) && H >= 1 && KVH >= 1 && H % KVH == 0);
  CHK(qkv.dim() == 3 && qkv.size(2) == (H + 2 * KVH) * hd && qkv.numel() > 0);
  const int64_t B = qkv.size(0), S = qkv.size(1), S32 = (S + 31) / 32 * 32;
  CHK(cos.size(-1) == hd / 2 && cos.numel() > 0 && cos.numel() <= INT_MAX && sin.sizes() == cos.sizes() && (positions.numel() == S || positions.numel() == B * S));
  CHK((((size_t)qkv.data_ptr() | (size_t)cos.data_ptr() | (size_t)sin.data_ptr()) & 15) == 0);
  CHK(B <= 65535 && H + 2 * KVH <= 65535 && B * S * (H + 2 * KVH) <= INT_MAX / 4);
  TrainArgs a{};
  a.qkv = P<bf16_t>(qkv);
  a.cos = cos.data_ptr<float>();
  a.sin = sin.data_ptr<float>();
  a.positions = positions.data_ptr<int>();
  a.B = (int)B;
  a.S = (int)S;
  a.S32 = (int)S32;
  a.H = (int)H;
  a.KVH = (int)KVH;
  a.per_row = positions.numel() == B * S && B > 1;
  a.places = (int)(cos.numel() / (hd / 2));
  a.scale = 1.f / sqrtf((float)hd);
  return a;
}

// -> out bf16 [B, S, H hd]; kept for the gradients: the packed projections by rows and
// transposed, out in fp32, the rows' sums of exponentials
std::vector<Tensor> train_attention(Tensor qkv, Tensor cos, Tensor sin, Tensor positions, int64_t H, int64_t KVH, int64_t hd) {
  auto a = train_args(qkv, cos, sin, positions, H, KVH, hd);
  auto r = torch::empty({a.B, H + 2 * KVH, a.S32, hd}, qkv.options()), t = torch::empty_like(r);
  auto out = torch::empty({a.B, a.S, H * hd}, qkv.options());
  auto o = f32(qkv, {a.B, a.S, H * hd}), lse = f32(qkv, {a.B, H, a.S32});
  a.r = M<bf16_t>(r);
  a.t = M<bf16_t>(t);
  a.out = M<bf16_t>(out);
  a.o = M<float>(o);
  a.lse = M<float>(lse);
  const int tiles = a.S32 / 32;
  const dim3 pack(tiles, a.H + 2 * a.KVH, a.B), walk((a.B * a.H * tiles + 3) / 4);
#define GO(HD_)                                                                                 \
  hipLaunchKernelGGL((pack_qkv_kernel<HD_>), pack, dim3(256), 0, cur_stream(), a);              \
  hipLaunchKernelGGL((train_forward_kernel<HD_>), walk, dim3(256), 0, cur_stream(), a);
  if (hd == 128) { GO(128) } else { GO(64) }
#undef GO
  return {out, r, t, o, lse};
}

Tensor train_attention_backward(Tensor dout, Tensor qkv, Tensor r, Tensor t, Tensor o, Tensor lse, Tensor cos, Tensor sin,
                                Tensor positions, int64_t H, int64_t KVH, int64_t hd) {
  auto a = train_args(qkv, cos, sin, positions, H, KVH, hd);
  check_io(dout, torch::kBFloat16);
  CHK(((size_t)dout.data_ptr() & 15) == 0 && dout.numel() == (int64_t)a.B * a.S * H * hd);
  for (const Tensor* x : {&r, &t}) { check_io(*x, torch::kBFloat16); CHK(x->numel() == (int64_t)a.B * (H + 2 * KVH) * a.S32 * hd); }
  for (const Tensor* x : {&o, &lse}) check_io(*x, torch::kFloat32);
  CHK(o.numel() == dout.numel() && lse.numel() == (int64_t)a.B * H * a.S32);
  auto dr = torch::empty({a.B, H, a.S32, hd}, qkv.options()), dt = torch::empty_like(dr), dqkv = torch::empty_like(qkv);
  auto delta = torch::empty_like(lse);
  a.r = M<bf16_t>(r);
  a.t = M<bf16_t>(t);
  a.o = M<float>(o);
  a.lse = M<float>(lse);
  a.dout = P<bf16_t>(dout);
  a.dr = M<bf16_t>(dr);
  a.dt = M<bf16_t>(dt);
  a.delta = M<float>(delta);
  a.dqkv = M<bf16_t>(dqkv);
  const int tiles = a.S32 / 32;
  const dim3 pack(tiles, a.H, a.B), queries((a.B * a.H * tiles + 3) / 4), keys128(a.B * a.KVH * ((tiles + 1) / 2)), keys64(a.B * a.KVH * tiles);
  if (hd == 128) {
    hipLaunchKernelGGL((pack_dout_kernel<128>), pack, dim3(256), 0, cur_stream(), a);
    hipLaunchKernelGGL((train_dkv_kernel<128, 2, 2, 2>), keys128, dim3(256), 0, cur_stream(), a);
    hipLaunchKernelGGL((train_dq_kernel<128>), queries, dim3(256), 0, cur_stream(), a);
  } else {
    hipLaunchKernelGGL((pack_dout_kernel<64>), pack, dim3(256), 0, cur_stream(), a);
    hipLaunchKernelGGL((train_dkv_kernel<64, 1, 2, 4>), keys64, dim3(512), 0, cur_stream(), a);
    hipLaunchKernelGGL((train_dq_kernel<64>), queries, dim3(256), 0, cur_stream(), a);
  }
  return dqkv;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("train_attention", &train_attention);
  m.def("train_attention_backward", &train_attention_backward);
}
