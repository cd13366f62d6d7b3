// A decode step's attention from the projection to the heads' outputs (head dim 64 or
// 128): norms and rotation of queries and the new key, append to both copies of the
// cache, GQA attention over the fragment-packed one
// (the reference: general_mha.py:78-106, 211-215).
//
// What bounds it is the cache's way from memory at many rows, and launches and single
// waves' chains at few: so there is one kernel where a block can take a whole row, and
// a short one that merges where rows are long and few. A block has a key head of a row
// (or a part of it), its waves take 32 positions in turn and merge in LDS. Scores are
// computed transposed from key rows in an order in which the lane that holds a head's
// probabilities feeds them to the value product. Parts are cut by the row's own
// length, so that short rows of a ragged batch have as many blocks as long ones.
//
// Probabilities of 64-channel heads stay fp32, as three bf16 parts that hold all their
// bits (errors against 64 bits 0.00164, 0.00188 with rounded ones); those of 128-channel
// heads are rounded to bf16 (0.00192 to 0.00197).
//
// The projection may come as fp32 sums over parts of k (tile_ops.hip): a block adds up
// its heads' numbers in LDS, which saves a kernel between the two: 2.4 us of its 4.7 in
// every layer (8 rows through 28 layers of 3584: 3285 to 3215 us).
#include "common.h"

struct DecodeArgs {
  const bf16_t* qkv;  // [B, (H + 2 KVH) HD]
  const float *cos, *sin;
  const int *positions, *lens;
  const bf16_t *qn, *kn;  // norms per head, or null
  bf16_t *kc, *vc, *kp, *vp, *out;
  const float* sums;   // or [nsums, B, (H + 2 KVH) HD], to be added up with bias
  const bf16_t* bias;
  int nsums;
  float *part, *ml;  // [B H][splits][HD], [B H][splits][2]
  int B, H, KVH, T, T32, npos, splits, places;  // places: rows of the rotation's tables
  float scale, eps;  // scale times log2 e
};

// Where the rotation's tables are read: a parked row may stand past their end
DEVINL size_t angle_row(const DecodeArgs& a, int pos) { return (size_t)min(max(pos, 0), a.places - 1); }

typedef __attribute__((ext_vector_type(4))) unsigned int uintx4;

DEVINL float lane_max(float v, int mask) { return fmaxf(v, __shfl_xor(v, mask)); }

// The new key and value of a key head, by one wave: normed and rotated, to the plain
// cache [B, KVH, T, HD] and the packed one.
template <int HD>
DEVINL void append(const DecodeArgs& a, int b, int kvh, int pos, int lane, const bf16_t* k, const bf16_t* v) {
  constexpr int HALF = HD / 2;
  const size_t head = (size_t)b * a.KVH + kvh;
  const bool on = lane < HALF;
  float x1 = on ? ld(k + lane) : 0.f, x2 = on ? ld(k + lane + HALF) : 0.f;
  if (a.kn) {
    const float inv = rsqrtf(wave_sum(x1 * x1 + x2 * x2) / (float)HD + a.eps);
    if (on) {
      x1 *= inv * ld(a.kn + lane);
      x2 *= inv * ld(a.kn + lane + HALF);
    }
  }
  bf16_t* kp = a.kp + (head * (a.T32 >> 4) + (pos >> 4)) * (HD / 32 * 512);
  bf16_t *kc = a.kc + (head * a.T + pos) * HD, *vc = a.vc + (head * a.T + pos) * HD;
  if (on) {
    const size_t at = angle_row(a, pos) * HALF + lane;
    const float c = a.cos[at], s = a.sin[at];
    const bf16_t r[2] = {f2b(x1 * c - x2 * s), f2b(x2 * c + x1 * s)};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int d = lane + i * HALF;
      kc[d] = r[i];
      kp[(d >> 5) * 512 + (((d & 31) >> 3) * 16 + (pos & 15)) * 8 + (d & 7)] = r[i];
    }
  }
#pragma unroll
  for (int d = lane; d < HD; d += 64) {
    vc[d] = v[d];
    a.vp[((head * (HD / 16) + (d >> 4)) * (a.T32 >> 5) + (pos >> 5)) * 512 + (((pos & 31) >> 3) * 16 + (d & 15)) * 8 + (pos & 7)] = v[d];
  }
}

// What a row's projection holds for the heads of a key head, as bf16: rep queries, key, value
template <int HD, int WAVES>
DEVINL void add_up(const DecodeArgs& a, int b, int kvh, int rep, bf16_t* own) {
  const size_t width = (size_t)(a.H + 2 * a.KVH) * HD, stride = a.B * width;
  for (int i = threadIdx.x * 4; i < (rep + 2) * HD; i += WAVES * 256) {
    const int slot = i / HD;
    const size_t at = (size_t)(slot < rep ? kvh * rep + slot : a.H + (slot - rep) * a.KVH + kvh) * HD + i % HD;
    const floatx4 v = sum_parts(a.sums, b * width + at, stride, a.nsums);
    float y[4], c[4] = {};
    if (a.bias) ld4(a.bias + at, c);
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = v[r] + c[r];
    st4(own + i, y);
  }
}

// Blocks of four waves, four a SIMD: with the three that it takes otherwise the 1024 blocks of 128
// rows and 8 key heads make a second round (us: 531 positions, 64 heads 57.5, 55.3; 100 to
// 270, 32 heads 31.5, 28.5; 64 channels, 64 to 128 rows of 200 to 700 positions, 20.8, 20.2).
// Of eight waves the code is the same either way.
template <int HD, int WAVES, bool SUMS>
__global__ __launch_bounds__(WAVES * 64, WAVES == 4 ? 4 : 2) void decode_attn_kernel(DecodeArgs a) {
  constexpr int KC = HD / 32, VG = HD / 16, HALF = HD / 2, ROW = HD + 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];  // [WAVES][rep][ROW] outputs
  __shared__ float lm[WAVES][16], ll[WAVES][16];
  __shared__ __attribute__((aligned(16))) bf16_t own_rows[SUMS ? 18 * HD : 1];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, quad = lane >> 4, rep = a.H / a.KVH;
  const int bh = blockIdx.x % (a.B * a.KVH), split = blockIdx.x / (a.B * a.KVH), b = bh / a.KVH, kvh = bh % a.KVH;
  const int pos = a.positions[a.npos > 1 ? b : 0], len = min(a.lens[b], a.T32);
  const int tiles = (len + 31) >> 5, t0 = tiles * split / a.splits, t1 = tiles * (split + 1) / a.splits;
  // the wave that reads the new position's tile appends it first; where none does (a
  // parked row), the first one
  const int own = pos < len ? pos >> 5 : -1;
  const bool fits = pos >= 0 && pos < a.T;
  const bool appends = fits && (own >= t0 && own < t1 ? (own - t0) % WAVES == wave : own < 0 && split == 0 && wave == 0);
  const bf16_t *q0, *k0, *v0;  // this key head's queries, key and value
  if (SUMS) {
    add_up<HD, WAVES>(a, b, kvh, rep, own_rows);
    __syncthreads();
    q0 = own_rows;
    k0 = own_rows + rep * HD;
    v0 = k0 + HD;
  } else {
    q0 = a.qkv + ((size_t)b * (a.H + 2 * a.KVH) + (size_t)kvh * rep) * HD;
    k0 = a.qkv + ((size_t)b * (a.H + 2 * a.KVH) + a.H + kvh) * HD;
    v0 = k0 + (size_t)a.KVH * HD;
  }
  if (appends) {
    append<HD>(a, b, kvh, pos, lane, k0, v0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  // this lane's query head, normed and rotated: dims c * 32 + quad * 8 + 0..7
  bf16x8 qf[KC];
  {
    const bf16_t* q = q0 + min(col, rep - 1) * HD + quad * 8;
    float x[KC][8], inv = 1.f;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      ld4(q + c * 32, x[c]);
      ld4(q + c * 32 + 4, x[c] + 4);
    }
    if (a.qn) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) ss += x[c][j] * x[c][j];
      ss += __shfl_xor(ss, 16);
      ss += __shfl_xor(ss, 32);
      inv = rsqrtf(ss / (float)HD + a.eps);
#pragma unroll
      for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) x[c][j] *= inv * ld(a.qn + c * 32 + quad * 8 + j);
    }
#pragma unroll
    for (int c = 0; c < KC / 2; ++c) {
      const size_t at = angle_row(a, pos) * HALF + c * 32 + quad * 8;
      const float *cs = a.cos + at, *sn = a.sin + at;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x1 = x[c][j], x2 = x[c + KC / 2][j];
        qf[c][j] = (__bf16)(x1 * cs[j] - x2 * sn[j]);
        qf[c + KC / 2][j] = (__bf16)(x2 * cs[j] + x1 * sn[j]);
      }
    }
  }
  float m = -1e30f;
  floatx4 o[VG], l = (floatx4)(0.f);  // l: the same sum in all four
  bf16x8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.f;
#pragma unroll
  for (int g = 0; g < VG; ++g) o[g] = (floatx4)(0.f);
  // key rows of the two products of 16: row i is position i / 4 * 8 + i % 4, and 4 more
  const int p = (col >> 2) * 8 + (col & 3);
  const bf16_t* kb = a.kp + (size_t)bh * a.T32 * HD + (p >> 4) * (KC * 512) + (quad * 16 + (p & 15)) * 8;
  const bf16_t* vb = a.vp + (size_t)bh * a.T32 * HD + lane * 8;
  for (int t = t0 + wave; t < t1; t += WAVES) {
    bf16x8 kf[2][KC], vf[VG];
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
        kf[hf][c] = __builtin_nontemporal_load((const bf16x8*)(kb + (size_t)t * (HD * 32) + c * 512 + hf * 32));
#pragma unroll
    for (int g = 0; g < VG; ++g)
      vf[g] = __builtin_nontemporal_load((const bf16x8*)(vb + ((size_t)g * (a.T32 >> 5) + t) * 512));
    floatx4 sc[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      sc[hf] = (floatx4)(0.f);
#pragma unroll
      for (int c = 0; c < KC; ++c) sc[hf] = mma(kf[hf][c], qf[c], sc[hf]);
    }
    float v[8], top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = t * 32 + quad * 8 + i < len ? sc[i >> 2][i & 3] * a.scale : -INFINITY;
      top = fmaxf(top, v[i]);
    }
    if (__any(top > m)) {
      top = fmaxf(m, lane_max(lane_max(top, 16), 32));
      const float f = __builtin_amdgcn_exp2f(m - top);
      m = top;
      l *= f;
#pragma unroll
      for (int g = 0; g < VG; ++g) o[g] *= f;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __builtin_amdgcn_exp2f(v[i] - m);
    if constexpr (HD == 64) {
      bf16x8 pf[3];
      split3(v, pf);
      l = mma3(ones, pf, l);
#pragma unroll
      for (int g = 0; g < VG; ++g) o[g] = mma3(vf[g], pf, o[g]);
    } else {
      bf16x8 pf;
#pragma unroll
      for (int i = 0; i < 8; ++i) pf[i] = (__bf16)v[i];
      l = mma(ones, pf, l);
#pragma unroll
      for (int g = 0; g < VG; ++g) o[g] = mma(vf[g], pf, o[g]);
    }
  }
  if (quad == 0) {
    lm[wave][col] = m;
    ll[wave][col] = l[0];
  }
  if (col < rep)
#pragma unroll
    for (int g = 0; g < VG; ++g) *(floatx4*)(lds + (wave * rep + col) * ROW + g * 16 + quad * 4) = o[g];
  __syncthreads();
  for (int i = threadIdx.x * 4; i < rep * HD; i += WAVES * 256) {
    const int h = i / HD, d = i % HD;
    float top = lm[0][h], sum = 0.f;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, lm[w][h]);
    floatx4 r = (floatx4)(0.f);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(lm[w][h] - top);
      sum += f * ll[w][h];
      r += f * *(const floatx4*)(lds + (w * rep + h) * ROW + d);
    }
    const size_t row = (size_t)b * a.H + kvh * rep + h;
    if (a.splits > 1) {
      *(floatx4*)(a.part + (row * a.splits + split) * HD + d) = r;
      if (d == 0) {
        a.ml[(row * a.splits + split) * 2] = top;
        a.ml[(row * a.splits + split) * 2 + 1] = sum;
      }
    } else {
      const float f = sum > 0.f ? 1.f / sum : 0.f;
      float y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = r[j] * f;
      st4(a.out + row * HD + d, y);
    }
  }
}

// A wave a head of a row: up to 64 parts, weighed by how far their maxima lie below
// the largest; four parts at a time.
template <int HD>
__global__ __launch_bounds__(256) void decode_merge_kernel(DecodeArgs a) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= a.B * a.H) return;
  const float* ml = a.ml + (size_t)row * a.splits * 2;
  const bool in = lane < a.splits;
  const float mine = in ? ml[lane * 2] : -1e30f;
  float top = mine;
#pragma unroll
  for (int mask = 1; mask < 64; mask <<= 1) top = lane_max(top, mask);
  const float f = in ? __builtin_amdgcn_exp2f(mine - top) : 0.f, sum = wave_sum(in ? f * ml[lane * 2 + 1] : 0.f);
  float o[HD / 64] = {};
  const float* part = a.part + (size_t)row * a.splits * HD + lane;
  for (int s = 0; s < a.splits; s += 4) {
    float v[4][HD / 64];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < HD / 64; ++i) v[k][i] = part[(size_t)min(s + k, a.splits - 1) * HD + i * 64];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float by = __shfl(f, min(s + k, 63));  // 0 past the last part
#pragma unroll
      for (int i = 0; i < HD / 64; ++i) o[i] += by * v[k][i];
    }
  }
#pragma unroll
  for (int i = 0; i < HD / 64; ++i) st(a.out + (size_t)row * HD + i * 64 + lane, sum == 0.f ? 0.f : o[i] / sum);  // NaN stays
}

// ===========================================================================
// host side
// ===========================================================================

template <int HD>
static void run_decode(DecodeArgs a, const Tensor& qkv) {
  const int heads = a.B * a.KVH, rep = a.H / a.KVH, tiles = a.T32 / 32;
  // eight waves a block where blocks are few. A block takes a whole row while its waves
  // have 4 tiles of 32 positions each or there are blocks enough; else some 256 blocks
  // with 2 tiles a wave at least
  const int waves = heads < 512 ? 8 : 4;
  a.splits = heads >= 512 || tiles <= 4 * waves ? 1 : std::max(1, std::min({(256 + heads - 1) / heads, tiles / (2 * waves), 64}));
  Tensor part, ml;
  if (a.splits > 1) {
    part = f32(qkv, {(int64_t)a.B * a.H, a.splits, HD});
    ml = f32(qkv, {(int64_t)a.B * a.H, a.splits, 2});
    a.part = part.data_ptr<float>();
    a.ml = ml.data_ptr<float>();
  }
  const int lds = waves * rep * (HD + 4) * (int)sizeof(float);
  auto run = [&](auto kernel) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    TORCH_CHECK(e == hipSuccess, "no LDS for attention outputs");
    hipLaunchKernelGGL(kernel, dim3(heads * a.splits), dim3(waves * 64), lds, cur_stream(), a);
  };
  if (a.sums) {
    if (waves == 8) run(decode_attn_kernel<HD, 8, true>);
    else run(decode_attn_kernel<HD, 4, true>);
  } else if (waves == 8) run(decode_attn_kernel<HD, 8, false>);
  else run(decode_attn_kernel<HD, 4, false>);
  if (a.splits > 1)
    hipLaunchKernelGGL((decode_merge_kernel<HD>), dim3((a.B * a.H + 3) / 4), dim3(256), 0, cur_stream(), a);
}

// qkv [B, 1, (H + 2 KVH) HD] as projected (left as it is; not read where sums
// [n, B, (H + 2 KVH) HD], fp32, and their bias take its place); kc, vc [B, KVH, T, HD];
// kp, vp their packed copies; lens: positions that rows see, the new one included.
// -> [B, 1, H HD]
Tensor decode_attend(Tensor qkv, Tensor cos, Tensor sin, Tensor positions, Tensor lens, Tensor kc, Tensor vc, Tensor kp,
                     Tensor vp, int64_t heads, int64_t kv_heads, OptT q_norm, OptT k_norm, double eps, OptT sums, OptT bias) {
  check_io(qkv, torch::kBFloat16);
  for (const Tensor* t : {&kc, &vc, &kp, &vp}) {
    check_io(*t, torch::kBFloat16);
    CHK(((size_t)t->data_ptr() & 15) == 0 && t->size(0) >= qkv.size(0));
  }
  check_io(cos, torch::kFloat32);
  check_io(sin, torch::kFloat32);
  check_io(positions, torch::kInt32);
  check_io(lens, torch::kInt32);
  DecodeArgs a{};
  a.B = (int)qkv.size(0);
  a.H = (int)heads;
  a.KVH = (int)kv_heads;
  CHK(qkv.dim() == 3 && qkv.size(1) == 1 && a.B >= 1 && kv_heads >= 1 && heads % kv_heads == 0 && heads / kv_heads <= 16);
  const int HD = (int)kc.size(3);
  CHK((HD == 64 || HD == 128) && qkv.size(2) == (heads + 2 * kv_heads) * HD && ((size_t)qkv.data_ptr() & 7) == 0);
  a.T = (int)kc.size(2);
  a.T32 = (int)kp.size(2) * 16;
  CHK(kc.size(1) == kv_heads && vc.sizes() == kc.sizes() && a.T <= a.T32 && a.T32 % 32 == 0);
  CHK(kp.numel() == kp.size(0) * kv_heads * a.T32 * HD && vp.numel() == vp.size(0) * kv_heads * a.T32 * HD);
  CHK(cos.size(-1) == HD / 2 && cos.numel() > 0 && cos.numel() <= INT_MAX && sin.sizes() == cos.sizes());
  a.places = (int)(cos.numel() / (HD / 2));
  a.npos = (int)positions.numel();
  CHK((a.npos == 1 || a.npos == a.B) && lens.numel() >= a.B);
  CHK((int64_t)a.B * kv_heads * 64 <= INT_MAX);
  for (const OptT* n : {&q_norm, &k_norm})
    if (*n) { check_io(**n, torch::kBFloat16); CHK((*n)->numel() == HD); }
  a.qn = q_norm ? P<bf16_t>(*q_norm) : nullptr;
  a.kn = k_norm ? P<bf16_t>(*k_norm) : nullptr;
  a.qkv = P<bf16_t>(qkv);
  if (sums) {
    check_io(*sums, torch::kFloat32);
    CHK(sums->dim() == 3 && sums->size(0) >= 1 && sums->size(0) <= 1024 && sums->numel() == sums->size(0) * qkv.numel());
    CHK(sums->size(1) == a.B && ((size_t)sums->data_ptr() & 15) == 0);
    a.sums = sums->data_ptr<float>();
    a.nsums = (int)sums->size(0);
    if (bias) {
      check_io(*bias, torch::kBFloat16);
      CHK(bias->numel() == qkv.size(2) && ((size_t)bias->data_ptr() & 7) == 0);
      a.bias = P<bf16_t>(*bias);
    }
  }
  a.cos = cos.data_ptr<float>();
  a.sin = sin.data_ptr<float>();
  a.positions = positions.data_ptr<int>();
  a.lens = lens.data_ptr<int>();
  a.kc = M<bf16_t>(kc);
  a.vc = M<bf16_t>(vc);
  a.kp = M<bf16_t>(kp);
  a.vp = M<bf16_t>(vp);
  a.eps = (float)eps;
  a.scale = 1.4426950408889634f / sqrtf((float)HD);
  auto out = torch::empty({a.B, 1, heads * HD}, qkv.options());
  a.out = M<bf16_t>(out);
  if (HD == 128) run_decode<128>(a, qkv);
  else run_decode<64>(a, qkv);
  return out;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("decode_attend", &decode_attend, pybind11::arg("qkv"), pybind11::arg("cos"), pybind11::arg("sin"),
        pybind11::arg("positions"), pybind11::arg("lens"), pybind11::arg("kc"), pybind11::arg("vc"), pybind11::arg("kp"),
        pybind11::arg("vp"), pybind11::arg("heads"), pybind11::arg("kv_heads"), pybind11::arg("q_norm"),
        pybind11::arg("k_norm"), pybind11::arg("eps"), pybind11::arg("sums") = pybind11::none(),
        pybind11::arg("bias") = pybind11::none());
}
