// What lies between a training pass's matrix products, bf16 tensors with fp32
// arithmetic: gradients of the norms and of the gated activation, and the way from a
// fused projection to attention's fp32 heads and back (the reference leaves training
// to torch's operators; its decoder's are general_mha.py:83-226, llm_utils.py:465-500).
//
// All of it is bound by memory: every tensor is read once and written once, where
// separate operators passed fp32 copies of it through memory some ten times.
#include "common.h"

DEVINL void st8(bf16_t* p, const float* o) {
  bf16x8 v;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (__bf16)o[i];
  *(bf16x8*)p = v;
}

// ---------------------------------------------------------------------------
// y = f / rms(f) (w + add) with f = x, or x + res (whose bf16 sum s is an output too):
//   df = ds + (dn - n mean(dn n)) / rms,  n = f / rms,  dn = dy (w + add)
// A block walks rows and keeps its share of dw = sum dy n in registers: [blocks, D]
// sums that a second kernel adds in order. 4096 rows of 4096: 25 us for 100 MB
// ---------------------------------------------------------------------------
template <int NC, bool DW>
__global__ __launch_bounds__(256) void norm_backward_kernel(
    const bf16_t* __restrict__ dy, const bf16_t* __restrict__ ds, const bf16_t* __restrict__ x,
    const bf16_t* __restrict__ res, const bf16_t* __restrict__ w, bf16_t* __restrict__ dx, float* __restrict__ dw_part,
    int rows, int D, float eps, float add) {
  __shared__ float red[2][2][4];  // alternating: a row's sums are read while the next are written
  float dw[DW ? NC * 8 : 1];
  if (DW)
#pragma unroll
    for (int i = 0; i < NC * 8; ++i) dw[i] = 0.f;
  int turn = 0;
  for (int row = blockIdx.x; row < rows; row += gridDim.x, turn ^= 1) {
    const size_t off = (size_t)row * D;
    float f[NC][8], g[NC][8], ss = 0.f, dot = 0.f;  // g: dy, then dy (w + add)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int i = (c * 256 + threadIdx.x) * 8;
      if (i >= D) break;
      float by[8];
      ld8(x + off + i, f[c]);
      if (res) {
        float r[8];
        ld8(res + off + i, r);
#pragma unroll
        for (int j = 0; j < 8; ++j) f[c][j] += r[j];
      }
      ld8(dy + off + i, g[c]);
      ld8(w + i, by);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        ss += f[c][j] * f[c][j];
        dot += f[c][j] * g[c][j] * (by[j] + add);
      }
    }
    ss = wave_sum(ss);
    dot = wave_sum(dot);
    if ((threadIdx.x & 63) == 0) {
      red[turn][0][threadIdx.x >> 6] = ss;
      red[turn][1][threadIdx.x >> 6] = dot;
    }
    __syncthreads();
    const float* s = red[turn][0];
    const float* d = red[turn][1];
    const float inv = rsqrtf((s[0] + s[1] + s[2] + s[3]) / (float)D + eps);
    const float mean = inv * inv * (d[0] + d[1] + d[2] + d[3]) / (float)D;  // mean(dn n) / rms(f)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int i = (c * 256 + threadIdx.x) * 8;
      if (i >= D) break;
      float by[8], o[8], more[8] = {};
      ld8(w + i, by);
      if (ds) ld8(ds + off + i, more);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (DW) dw[c * 8 + j] += g[c][j] * f[c][j] * inv;
        o[j] = more[j] + inv * (g[c][j] * (by[j] + add) - f[c][j] * mean);
      }
      st8(dx + off + i, o);
    }
  }
  if (DW)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int i = (c * 256 + threadIdx.x) * 8;
      if (i >= D) break;
#pragma unroll
      for (int j = 0; j < 8; j += 4) st4(dw_part + (size_t)blockIdx.x * D + i + j, dw + c * 8 + j);
    }
}

// dw of 64 columns a block: 16 waves share the parts, 8 loads on their way in each
// (512 parts of 2048 columns: 4.5 us; 39 by 4 waves with one load each)
__global__ __launch_bounds__(1024) void sum_columns_kernel(const float* __restrict__ part, bf16_t* __restrict__ dw, int parts, int D) {
  __shared__ float red[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (col < D) {
    int p = wave;
    for (; p + 7 * 16 < parts; p += 8 * 16) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = part[(size_t)(p + i * 16) * D + col];
#pragma unroll
      for (int i = 0; i < 8; ++i) s += v[i];
    }
    for (; p < parts; p += 16) s += part[(size_t)p * D + col];
  }
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && col < D) {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) sum += red[w][lane];
    st(dw + col, sum);
  }
}

// ---------------------------------------------------------------------------
// y = silu(gate) up on rows [gate | up]
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void swiglu_backward_kernel(const bf16_t* __restrict__ gu, const bf16_t* __restrict__ dy,
                                                              bf16_t* __restrict__ dgu, long long n8, int i8) {
  const long long stride = (long long)gridDim.x * 256;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n8; i += stride) {
    const long long row = i / i8, at = row * i8 * 16 + (i - row * i8) * 8;
    float g[8], u[8], d[8], dg[8], du[8];
    ld8(gu + at, g);
    ld8(gu + at + i8 * 8, u);
    ld8(dy + i * 8, d);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float s = sigmoidf(g[j]);
      du[j] = d[j] * g[j] * s;
      dg[j] = d[j] * u[j] * s * (1.f + g[j] * (1.f - s));
    }
    st8(dgu + at, dg);
    st8(dgu + at + i8 * 8, du);
  }
}

// ---------------------------------------------------------------------------
// projection [B, S, (H + 2 KVH) hd] -> fp32 [B, H, S, hd]: queries and keys rotated
// (rounded to bf16 as the operators' results are), keys and values repeated for every
// head that shares them; and the gradients' way back, repeated ones summed in fp32.
// A thread has 4 channels and their partners, hd / 2 further.
// ---------------------------------------------------------------------------
struct HeadArgs {
  const float *cos, *sin;
  const int* positions;
  int B, S, H, KVH, hd, per_row, places;  // per_row: positions [B, S], else [S]; places: rows of the tables
};

__global__ __launch_bounds__(256) void split_heads_kernel(const bf16_t* __restrict__ qkv, float* __restrict__ q,
                                                          float* __restrict__ k, float* __restrict__ v, HeadArgs a, long long n) {
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  if (i >= n) return;
  const int quads = a.hd / 8, slots = a.H + 2 * a.KVH, half = a.hd / 2;
  const int c = (int)(i % quads) * 4, slot = (int)(i / quads % slots);
  const long long tok = i / quads / slots;
  const int s = (int)(tok % a.S), b = (int)(tok / a.S);
  const bf16_t* src = qkv + (tok * slots + slot) * a.hd + c;
  float x1[4], x2[4];
  ld4(src, x1);
  ld4(src + half, x2);
  if (slot < a.H + a.KVH) {
    float co[4], si[4];
    const int pos = table_row(a.positions[a.per_row ? tok : s], a.places);
    ld_angles(a.cos, pos, half, c, co);
    ld_angles(a.sin, pos, half, c, si);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float y1 = x1[j] * co[j] - x2[j] * si[j], y2 = x2[j] * co[j] + x1[j] * si[j];
      x1[j] = rounded(y1);
      x2[j] = rounded(y2);
    }
  }
  const int rep = a.H / a.KVH;
  float* dst = slot < a.H ? q : slot < a.H + a.KVH ? k : v;
  const int h0 = slot < a.H ? slot : (slot - a.H) % a.KVH * rep, times = slot < a.H ? 1 : rep;
  for (int r = 0; r < times; ++r) {
    float* o = dst + (((size_t)b * a.H + h0 + r) * a.S + s) * a.hd + c;
    st4(o, x1);
    st4(o + half, x2);
  }
}

__global__ __launch_bounds__(256) void split_heads_backward_kernel(const float* __restrict__ dq, const float* __restrict__ dk,
                                                                   const float* __restrict__ dv, bf16_t* __restrict__ dqkv,
                                                                   HeadArgs a, long long n) {
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  if (i >= n) return;
  const int quads = a.hd / 8, slots = a.H + 2 * a.KVH, half = a.hd / 2;
  const int c = (int)(i % quads) * 4, slot = (int)(i / quads % slots);
  const long long tok = i / quads / slots;
  const int s = (int)(tok % a.S), b = (int)(tok / a.S), rep = a.H / a.KVH;
  const float* src = slot < a.H ? dq : slot < a.H + a.KVH ? dk : dv;
  const int h0 = slot < a.H ? slot : (slot - a.H) % a.KVH * rep, times = slot < a.H ? 1 : rep;
  float g1[4] = {}, g2[4] = {};
  for (int r = 0; r < times; ++r) {
    const float* p = src + (((size_t)b * a.H + h0 + r) * a.S + s) * a.hd + c;
    float t1[4], t2[4];
    ld4(p, t1);
    ld4(p + half, t2);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      g1[j] += t1[j];
      g2[j] += t2[j];
    }
  }
  if (slot < a.H + a.KVH) {
    float co[4], si[4];
    const int pos = table_row(a.positions[a.per_row ? tok : s], a.places);
    ld_angles(a.cos, pos, half, c, co);
    ld_angles(a.sin, pos, half, c, si);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float y1 = rounded(g1[j]), y2 = rounded(g2[j]);
      g1[j] = y1 * co[j] + y2 * si[j];
      g2[j] = y2 * co[j] - y1 * si[j];
    }
  }
  bf16_t* dst = dqkv + (tok * slots + slot) * a.hd + c;
  st4(dst, g1);
  st4(dst + half, g2);
}

// fp32 [B, H, S, hd] <-> bf16 [B, S, H hd]
template <bool TO_TOKENS>
__global__ __launch_bounds__(256) void heads_kernel(const void* __restrict__ src, void* __restrict__ dst, int S, int H, int hd,
                                                    long long n) {
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  if (i >= n) return;
  const int quads = hd / 4, c = (int)(i % quads) * 4, h = (int)(i / quads % H);
  const long long tok = i / quads / H;
  const size_t heads = (((size_t)(tok / S) * H + h) * S + tok % S) * hd + c, tokens = ((size_t)tok * H + h) * hd + c;
  float v[4];
  if (TO_TOKENS) {
    ld4((const float*)src + heads, v);
    st4((bf16_t*)dst + tokens, v);
  } else {
    ld4((const bf16_t*)src + tokens, v);
    st4((float*)dst + heads, v);
  }
}

// ===========================================================================
// host side
// ===========================================================================

static void check_16(const Tensor& t, torch::ScalarType dt) {
  check_io(t, dt);
  CHK(((size_t)t.data_ptr() & 15) == 0);
}

// -> dx (of x and, given, res), and dw where asked
std::vector<Tensor> norm_backward(Tensor dy, OptT ds, Tensor x, OptT res, Tensor w, double eps, double add, bool need_dw) {
  for (const Tensor& t : {dy, x, w}) check_16(t, torch::kBFloat16);
  const int64_t D = x.size(-1), rows = x.numel() / D;
  CHK(D % 8 == 0 && D <= 16384 && dy.numel() == x.numel() && w.numel() == D && rows <= INT_MAX);
  for (const OptT* t : {&ds, &res})
    if (*t) { check_16(**t, torch::kBFloat16); CHK((*t)->numel() == x.numel()); }
  auto dx = torch::empty_like(x);
  const int blocks = (int)std::min<int64_t>(rows, need_dw ? 512 : INT_MAX);
  Tensor part, dw;
  if (need_dw) {
    part = f32(x, {std::max(blocks, 1), D});
    dw = rows ? torch::empty_like(w) : torch::zeros_like(w);
  }
  if (rows) {
    auto run = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, cur_stream(), P<bf16_t>(dy), ds ? P<bf16_t>(*ds) : nullptr,
                         P<bf16_t>(x), res ? P<bf16_t>(*res) : nullptr, P<bf16_t>(w), M<bf16_t>(dx),
                         need_dw ? part.data_ptr<float>() : nullptr, (int)rows, (int)D, (float)eps, (float)add);
    };
#define GO(NC_) if (need_dw) run(norm_backward_kernel<NC_, true>); else run(norm_backward_kernel<NC_, false>);
    if (D <= 2048) { GO(1) }
    else if (D <= 4096) { GO(2) }
    else if (D <= 8192) { GO(4) }
    else { GO(8) }
#undef GO
    if (need_dw)
      hipLaunchKernelGGL(sum_columns_kernel, dim3((D + 63) / 64), dim3(1024), 0, cur_stream(), part.data_ptr<float>(),
                         M<bf16_t>(dw), blocks, (int)D);
  }
  if (need_dw) return {dx, dw};
  return {dx};
}

Tensor swiglu_backward(Tensor gu, Tensor dy) {
  check_16(gu, torch::kBFloat16);
  check_16(dy, torch::kBFloat16);
  CHK(gu.numel() == 2 * dy.numel() && gu.size(-1) == 2 * dy.size(-1) && dy.size(-1) % 8 == 0);
  auto dgu = torch::empty_like(gu);
  const long long n8 = dy.numel() / 8;
  if (n8)
    hipLaunchKernelGGL(swiglu_backward_kernel, dim3((unsigned)std::min<long long>((n8 + 255) / 256, 8192)), dim3(256), 0,
                       cur_stream(), P<bf16_t>(gu), P<bf16_t>(dy), M<bf16_t>(dgu), n8, (int)(dy.size(-1) / 8));
  return dgu;
}

static HeadArgs head_args(const Tensor& cos, const Tensor& sin, const Tensor& positions, int64_t B, int64_t S, int64_t H,
                          int64_t KVH, int64_t hd) {
  check_16(cos, torch::kFloat32);
  check_16(sin, torch::kFloat32);
  check_io(positions, torch::kInt32);
  CHK(H >= 1 && KVH >= 1 && H % KVH == 0 && hd % 8 == 0 && cos.size(-1) == hd / 2 && cos.numel() > 0 && cos.numel() <= INT_MAX && sin.sizes() == cos.sizes());
  CHK(positions.numel() == S || positions.numel() == B * S);
  CHK(B <= INT_MAX && S <= INT_MAX && B * S * (H + 2 * KVH) * (hd / 8) / 256 < INT_MAX);
  return HeadArgs{cos.data_ptr<float>(), sin.data_ptr<float>(), positions.data_ptr<int>(), (int)B, (int)S, (int)H, (int)KVH,
                  (int)hd, positions.numel() == B * S && B > 1, (int)(cos.numel() / (hd / 2))};
}

// -> q, k, v fp32 [B, H, S, hd]
std::vector<Tensor> split_heads(Tensor qkv, Tensor cos, Tensor sin, Tensor positions, int64_t H, int64_t KVH, int64_t hd) {
  check_16(qkv, torch::kBFloat16);
  CHK(qkv.dim() == 3 && qkv.size(2) == (H + 2 * KVH) * hd);
  const int64_t B = qkv.size(0), S = qkv.size(1);
  const auto a = head_args(cos, sin, positions, B, S, H, KVH, hd);
  Tensor o[3];
  for (Tensor& t : o) t = f32(qkv, {B, H, S, hd});
  const long long n = B * S * (H + 2 * KVH) * (hd / 8);
  if (n)
    hipLaunchKernelGGL(split_heads_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, cur_stream(), P<bf16_t>(qkv),
                       M<float>(o[0]), M<float>(o[1]), M<float>(o[2]), a, n);
  return {o[0], o[1], o[2]};
}

Tensor split_heads_backward(Tensor dq, Tensor dk, Tensor dv, Tensor cos, Tensor sin, Tensor positions, int64_t KVH) {
  for (const Tensor& t : {dq, dk, dv}) { check_16(t, torch::kFloat32); CHK(t.dim() == 4 && t.sizes() == dq.sizes()); }
  const int64_t B = dq.size(0), H = dq.size(1), S = dq.size(2), hd = dq.size(3);
  const auto a = head_args(cos, sin, positions, B, S, H, KVH, hd);
  auto out = torch::empty({B, S, (H + 2 * KVH) * hd}, dq.options().dtype(torch::kBFloat16));
  const long long n = B * S * (H + 2 * KVH) * (hd / 8);
  if (n)
    hipLaunchKernelGGL(split_heads_backward_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, cur_stream(),
                       P<float>(dq), P<float>(dk), P<float>(dv), M<bf16_t>(out), a, n);
  return out;
}

// fp32 [B, H, S, hd] -> bf16 [B, S, H hd]
Tensor merge_heads(Tensor o) {
  check_16(o, torch::kFloat32);
  CHK(o.dim() == 4 && o.size(3) % 4 == 0);
  const int64_t B = o.size(0), H = o.size(1), S = o.size(2), hd = o.size(3);
  auto out = torch::empty({B, S, H * hd}, o.options().dtype(torch::kBFloat16));
  const long long n = o.numel() / 4;
  CHK(n / 256 < INT_MAX);
  if (n)
    hipLaunchKernelGGL((heads_kernel<true>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, cur_stream(), o.data_ptr(),
                       out.data_ptr(), (int)S, (int)H, (int)hd, n);
  return out;
}

Tensor merge_heads_backward(Tensor d, int64_t H) {
  check_16(d, torch::kBFloat16);
  CHK(d.dim() == 3 && H >= 1 && d.size(2) % (4 * H) == 0);
  const int64_t B = d.size(0), S = d.size(1), hd = d.size(2) / H;
  auto out = f32(d, {B, H, S, hd});
  const long long n = d.numel() / 4;
  CHK(n / 256 < INT_MAX);
  if (n)
    hipLaunchKernelGGL((heads_kernel<false>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, cur_stream(), d.data_ptr(),
                       out.data_ptr(), (int)S, (int)H, (int)hd, n);
  return out;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("norm_backward", &norm_backward);
  m.def("swiglu_backward", &swiglu_backward);
  m.def("split_heads", &split_heads);
  m.def("split_heads_backward", &split_heads_backward);
  m.def("merge_heads", &merge_heads);
  m.def("merge_heads_backward", &merge_heads_backward);
}
