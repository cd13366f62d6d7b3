// Products of one or two rows (decode steps of so many sequences, prompts of so many
// tokens) with bf16 weights as they lie in the checkpoint, [N, K] row-major:
//   y = x W^T + bias, y = norm(x) W^T + bias, y = silu(norm(x) Wg^T) norm(x) Wu^T,
//   y = r + x W^T.
// (The reference runs these as separate modules, general_mha.py:83-102,
// llm_utils.py:465-500.)
//
// What bounds them is the weights' way from memory, and with small matrices the
// launches around it; so the norm before and the activation or the residual sum
// after a product belong to its kernel. A wave takes R weight rows at a time, 512
// numbers of each (one load of 1 KB a row, whole lines) two steps deep, and
// multiplies pairs of bf16 into fp32 sums; matrix instructions would have 14 or more
// columns idle and want the weights in another order. Waves of a block share a row
// group's k where there are few rows. Weights are read once: non-temporal.
// One row, against the library (us, TB/s): [128256, 2048] 75 (7.0) and 113,
// [37888, 3584] 42 (6.4) and 57, [3584, 18944] 24 (5.7) and 48, [3072, 2048] 4.4 and 12.
#include "common.h"

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) unsigned int uintx4;  // 8 bf16

struct RowsArgs {
  const void* x;       // [m, K] bf16, or fp32 before a norm
  const bf16_t* w;     // [N, K]; GATED: [2 N, K], gate rows first
  const bf16_t* norm;  // [K]
  const bf16_t* bias;  // [N] or null
  const void* res;     // [m, N], ADD
  void* y;
  int m, N, K, groups;
  float eps, norm_add;
};

enum RowsSource { PLAIN_X, NORM_BF16, NORM_F32 };
// ADD_x: type of the residual; the sum is of the other type (fp32 is what the next norm reads)
enum RowsEnd { STORE, GATED_STORE, ADD_BF16, ADD_F32 };

// Sums over the wave of COUNT (a power of two) values a lane each: every exchange
// halves what is left, so that this takes about COUNT shuffles and not 6 COUNT.
// Lane l ends with the sum of value l >> (6 - log2 COUNT).
template <int COUNT> struct Sums { typedef __attribute__((ext_vector_type(COUNT))) float V; };
template <int COUNT, int MASK = 32>
DEVINL float spread_sum(typename Sums<COUNT>::V v, int lane) {
  const bool up = lane & MASK;
  if constexpr (COUNT == 2) {
    float s = (up ? v[1] : v[0]) + __shfl_xor(up ? v[0] : v[1], MASK);
#pragma unroll
    for (int mask = MASK / 2; mask > 0; mask >>= 1) s += __shfl_xor(s, mask);
    return s;
  } else {
    typename Sums<COUNT / 2>::V h;
#pragma unroll
    for (int i = 0; i < COUNT / 2; ++i)
      h[i] = (up ? v[i + COUNT / 2] : v[i]) + __shfl_xor(up ? v[i] : v[i + COUNT / 2], MASK);
    return spread_sum<COUNT / 2, MASK / 2>(h, lane);
  }
}

// Values are rounded where the separate operators of many rows round; the order of the
// sums is these kernels' own, and another for one row than for two.
constexpr int MOST_X = 128 * 1024;  // bytes of normed rows

constexpr int log2_of(int n) { return n <= 1 ? 0 : 1 + log2_of(n / 2); }

// 16 bytes at `at` of a row of `bytes`, zeros where they lie past its end. AUX 2: read once.
template <int AUX>
DEVINL uintx4 load_row(const bf16_t* row, int bytes, int at) {
  return __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(
      __builtin_amdgcn_make_buffer_rsrc((void*)row, 0, bytes, 0x00027000), at, 0, AUX));
}

// M rows of x (a.m <= M of them real), R weight rows a wave at a time, KS waves of
// the block share a row group.
template <int M, int R, int KS, int SRC, int END>
__global__ __launch_bounds__(256) void rows_kernel(RowsArgs a) {
  constexpr bool TWO = END == GATED_STORE;
  constexpr int COUNT = M * R, SHIFT = 6 - log2_of(COUNT), PER = 4 / KS;  // row groups of a block
  typedef typename std::conditional<SRC == NORM_F32, float, bf16_t>::type X;
  extern __shared__ __attribute__((aligned(16))) bf16_t xs[];  // [m][K rounded up to 512], normed
  __shared__ float red[4][KS > 1 || SRC != PLAIN_X ? 64 : 1];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int ks = wave % KS, chunks = (a.K + 511) >> 9;
  const X* x = (const X*)a.x;
  // row r of a group, clamped: what lies past the end is not stored
  auto row_of = [&](int g, int r) {
    if (TWO) return min(g * (R / 2) + r % (R / 2), a.N - 1) + (r >= R / 2 ? a.N : 0);
    return min(g * R + r, a.N - 1);
  };
  // 512 numbers of the group's rows, and of x, from chunk c on: zeros past a row's end
  struct Part { uintx4 w[R], x[M]; };
  const int bytes = a.K * 2;
  auto load = [&](Part& p, int g, int c) {
    const int k = c * 1024 + lane * 16;
#pragma unroll
    for (int r = 0; r < R; ++r) p.w[r] = load_row<2>(a.w + (size_t)row_of(g, r) * a.K, bytes, k);
    if (SRC == PLAIN_X)
#pragma unroll
      for (int m = 0; m < M; ++m) p.x[m] = load_row<0>((const bf16_t*)a.x + (size_t)min(m, a.m - 1) * a.K, bytes, k);
  };
  const int n = chunks > ks ? (chunks - ks + KS - 1) / KS : 0;  // this wave's chunks
  // Numbers of x and of the norm's weights that a thread keeps: loads come back in order, so
  // that these go out before any weights. us, read behind the first weights, twice, and every
  // row group waited for by itself, and so: gate [16384, 2048] m 1 13.6, 12.9, m 2 15.1, 13.4; [9728, 896]
  // 7.2, 6.4; [4608, 3584] m 1 9.1, 8.8, m 2 11.2, 9.6
  constexpr int KEPT = SRC == PLAIN_X ? 0 : 2, RAW = sizeof(X) / 2;
  uintx4 kept[KEPT + 1][M][RAW], kept_by[KEPT + 1];
#pragma unroll
  for (int p = 0; p < KEPT; ++p) {
    const int i = min(p * 2048 + (int)threadIdx.x * 8, a.K - 8);
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int r = 0; r < RAW; ++r) kept[p][m][r] = ((const uintx4*)(x + (size_t)min(m, a.m - 1) * a.K + i))[r];
    kept_by[p] = *(const uintx4*)(a.norm + i);
  }
  __builtin_amdgcn_sched_barrier(0);
  // row m's numbers of piece p
  auto of_piece = [&](int p, int m, float* v) {
    if constexpr (SRC == NORM_F32)
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = __uint_as_float(kept[p][m][j / 4][j % 4]);
    else
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j * 2] = __uint_as_float(kept[p][m][0][j] << 16);
        v[j * 2 + 1] = __uint_as_float(kept[p][m][0][j] & 0xffff0000u);
      }
  };
  Part A, B;
  int g = blockIdx.x * PER + wave / KS;
  // Two chunks are on their way, with a norm, whose blocks have further row groups, also from one
  // group to the next
  int ahead_g = g, ahead = 0;
  auto load_next = [&](Part& p) {
    if (n == 0 || ahead_g - wave / KS >= a.groups) return;
    load(p, ahead_g, ks + ahead * KS);
    if (++ahead == n) {
      ahead = 0;
      ahead_g += gridDim.x * PER;
    }
  };
  // on their way while the rows of x are normed
  if (SRC != PLAIN_X) {
    load_next(A);
    load_next(B);
  } else {
    if (n > 0) load(A, g, ks);
    if (n > 1) load(B, g, ks + KS);
  }
  if (SRC != PLAIN_X) {
    float ss[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      ss[m] = 0.f;
#pragma unroll
      for (int p = 0; p < KEPT; ++p)
        if (p * 2048 + (int)threadIdx.x * 8 < a.K) {
          float v[8];
          of_piece(p, m, v);
#pragma unroll
          for (int j = 0; j < 8; ++j) ss[m] += v[j] * v[j];
        }
    }
    for (int i = KEPT * 2048 + threadIdx.x * 8; i < a.K; i += 2048)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        float v[8];
        ld8(x + (size_t)min(m, a.m - 1) * a.K + i, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) ss[m] += v[j] * v[j];
      }
#pragma unroll
    for (int m = 0; m < M; ++m) {
      ss[m] = wave_sum(ss[m]);
      if (lane == 0) red[wave][m] = ss[m];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; ++m) ss[m] = rsqrtf((red[0][m] + red[1][m] + red[2][m] + red[3][m]) / (float)a.K + a.eps);
    for (int i = a.K + threadIdx.x * 8; i < chunks * 512; i += 2048)
#pragma unroll
      for (int m = 0; m < M; ++m)
        if (m < a.m) *(uintx4*)(xs + m * chunks * 512 + i) = (uintx4)(0u);
    auto put = [&](int m, int i, const float* v, const float* by) {
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (__bf16)(v[j] * ss[m] * (by[j] + a.norm_add));
      *(bf16x8*)(xs + m * chunks * 512 + i) = o;
    };
#pragma unroll
    for (int p = 0; p < KEPT; ++p) {
      const int i = p * 2048 + (int)threadIdx.x * 8;
      if (i >= a.K) break;
      float by[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        by[j * 2] = __uint_as_float(kept_by[p][j] << 16);
        by[j * 2 + 1] = __uint_as_float(kept_by[p][j] & 0xffff0000u);
      }
#pragma unroll
      for (int m = 0; m < M; ++m) {
        if (m >= a.m) break;
        float v[8];
        of_piece(p, m, v);
        put(m, i, v, by);
      }
    }
    for (int i = KEPT * 2048 + threadIdx.x * 8; i < a.K; i += 2048) {
      float by[8];
      ld8(a.norm + i, by);
#pragma unroll
      for (int m = 0; m < M; ++m) {
        if (m >= a.m) break;
        float v[8];
        ld8(x + (size_t)m * a.K + i, v);
        put(m, i, v, by);
      }
    }
    __syncthreads();
  }
  // a row group, whose first chunk is in P
  auto group = [&](Part& P, Part& Q) {
    typename Sums<COUNT>::V acc = (typename Sums<COUNT>::V)(0.f);
    auto add = [&](Part& p, int i) {
      if (SRC != PLAIN_X)
#pragma unroll
        for (int m = 0; m < M; ++m)
          p.x[m] = *(const uintx4*)(xs + min(m, a.m - 1) * chunks * 512 + (ks + i * KS) * 512 + lane * 8);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int m = 0; m < M; ++m) {
            const unsigned w = p.w[r][j], x = p.x[m][j];
            acc[r * M + m] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), __builtin_bit_cast(bf16x2, x),
                                                             acc[r * M + m], false);
          }
    };
    int i = 0;
    if (SRC == PLAIN_X) {
      for (; i + 3 < n; i += 2) {
        add(P, i);
        load(P, g, ks + (i + 2) * KS);
        add(Q, i + 1);
        load(Q, g, ks + (i + 3) * KS);
      }
      if (n - i == 3) {
        add(P, i);
        load(P, g, ks + (i + 2) * KS);
        add(Q, i + 1);
        add(P, i + 2);
      } else if (n - i == 2) {
        add(P, i);
        add(Q, i + 1);
      } else if (n - i == 1) {
        add(P, i);
      }
    } else {
      for (; i + 1 < n; i += 2) {
        add(P, i);
        load_next(P);
        add(Q, i + 1);
        load_next(Q);
      }
      if (i < n) {
        add(P, i);
        load_next(P);
      }
    }
    float v = spread_sum<COUNT>(acc, lane);
    if (KS > 1) {
      if ((lane & ((1 << SHIFT) - 1)) == 0) red[wave][lane >> SHIFT] = v;
      __syncthreads();
      v = 0.f;
#pragma unroll
      for (int i = 0; i < KS; ++i) v += red[wave / KS * KS + i][lane >> SHIFT];
      __syncthreads();
    }
    const float other = TWO ? __shfl_xor(v, 32) : 0.f;
    const int idx = lane >> SHIFT, r = idx / M, m = idx % M;
    const int n = TWO ? g * (R / 2) + r : g * R + r;
    if (ks == 0 && (lane & ((1 << SHIFT) - 1)) == 0 && g < a.groups && m < a.m && n < a.N && (!TWO || lane < 32)) {
      const size_t o = (size_t)m * a.N + n;
      if (END == STORE) st((bf16_t*)a.y + o, v + (a.bias ? ld(a.bias + n) : 0.f));
      if (END == GATED_STORE) st((bf16_t*)a.y + o, siluf(rounded(v)) * rounded(other));
      if (END == ADD_BF16) ((float*)a.y)[o] = ld((const bf16_t*)a.res + o) + rounded(v);
      if (END == ADD_F32) st((bf16_t*)a.y + o, rounded(((const float*)a.res)[o]) + rounded(v));
    }
    g += gridDim.x * PER;
  };
  if (SRC == PLAIN_X) {  // blocks for all groups
    group(A, B);
    return;
  }
  // Waves that share k may have one an odd and one an even number of chunks, and then wait in different copies of
  // `group` for one another. The hardware's barrier counts a block's waves wherever they are, and each comes by
  // two of them a row group, of which all waves of a block have as many (g - wave / KS is the block's).
  while (g - wave / KS < a.groups) {
    group(A, B);
    if (n % 2 == 0 || g - wave / KS >= a.groups) continue;
    group(B, A);
  }
}

// ===========================================================================
// host side
// ===========================================================================

// Waves that share a row group: as many as it takes to have some 2000 waves that
// each keep a few KB in flight, fewer where the sums over the wave (4 or 8 exchanges
// a group and wave) would outweigh it. Measured, us for 1, 2, 4 waves a group and one
// row: [2048, 8192] 10.8, 8.3, 7.6; [3584, 18944] 23.9, 23.6, 24.1; two rows, [128256,
// 2048] 88, 77, 89. With a norm blocks also read all of x first, so that there are at
// most 512 or 1024 of them, which go on to further groups: one row, [3072, 2048] 6.1,
// 5.5, 5.5; [37888, 3584] 43.0, 42.1, 43.5.
template <int M, int KS, int SRC, int END>
static void launch_rows(const RowsArgs& a, int most) {
  const int lds = SRC == PLAIN_X ? 0 : a.m * ((a.K + 511) / 512) * 1024;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)rows_kernel<M, 4, KS, SRC, END>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, MOST_X);
    TORCH_CHECK(e == hipSuccess, "no LDS for the rows' norm");
  }
  const int blocks = (a.groups * KS + 3) / 4;
  hipLaunchKernelGGL((rows_kernel<M, 4, KS, SRC, END>), dim3(std::min(blocks, most)), dim3(256), lds, cur_stream(), a);
}

template <int M, int SRC, int END>
static void run_m(const RowsArgs& a) {
  if constexpr (SRC != PLAIN_X) {
    if (M == 1 || END == STORE) launch_rows<M, 2, SRC, END>(a, END == STORE ? 1024 : 512);
    else launch_rows<M, 1, SRC, END>(a, 512);
  } else {
    if (a.groups <= 4096 && a.K > 1536) launch_rows<M, 4, SRC, END>(a, INT_MAX);
    else launch_rows<M, 2, SRC, END>(a, INT_MAX);
  }
}

template <int SRC, int END>
static void run_rows(RowsArgs a) {
  const int per = END == GATED_STORE ? 2 : 4;
  a.groups = (a.N + per - 1) / per;
  if (a.m == 1) run_m<1, SRC, END>(a);
  else run_m<2, SRC, END>(a);
}

static RowsArgs rows_args(const Tensor& x, const Tensor& w, int64_t n) {
  check_io(w, torch::kBFloat16);
  CHK(x.is_cuda() && x.is_contiguous() && w.dim() == 2);
  RowsArgs a{};
  a.K = (int)w.size(1);
  CHK(a.K > 0 && a.K % 8 == 0 && x.size(-1) == a.K);
  a.m = (int)(x.numel() / a.K);
  CHK(a.m >= 1 && a.m <= 2 && n >= 1 && n <= INT_MAX / 16);
  a.N = (int)n;
  CHK(((size_t)x.data_ptr() & 15) == 0 && ((size_t)w.data_ptr() & 15) == 0);
  a.x = x.data_ptr();
  a.w = P<bf16_t>(w);
  return a;
}
static Tensor rows_out(const Tensor& x, int64_t n, torch::ScalarType dt) {
  auto shape = x.sizes().vec();
  shape.back() = n;
  return torch::empty(shape, x.options().dtype(dt));
}
static void take_norm(RowsArgs& a, const Tensor& norm, double eps, double add) {
  check_io(norm, torch::kBFloat16);
  CHK(norm.numel() == a.K && ((size_t)norm.data_ptr() & 15) == 0 && (int64_t)a.m * ((a.K + 511) / 512) * 1024 <= MOST_X);
  a.norm = P<bf16_t>(norm);
  a.eps = (float)eps;
  a.norm_add = (float)add;
}
static void take_bias(RowsArgs& a, const OptT& bias) {
  if (!bias) return;
  check_io(*bias, torch::kBFloat16);
  CHK(bias->numel() == a.N);
  a.bias = P<bf16_t>(*bias);
}

Tensor rows_linear(Tensor x, Tensor w, OptT bias) {
  check_io(x, torch::kBFloat16);
  auto a = rows_args(x, w, w.size(0));
  take_bias(a, bias);
  auto y = rows_out(x, a.N, torch::kBFloat16);
  a.y = y.data_ptr();
  run_rows<PLAIN_X, STORE>(a);
  return y;
}

Tensor rows_norm_linear(Tensor x, Tensor norm, double eps, double add, Tensor w, OptT bias) {
  check_io(x, torch::kBFloat16);
  auto a = rows_args(x, w, w.size(0));
  take_norm(a, norm, eps, add);
  take_bias(a, bias);
  auto y = rows_out(x, a.N, torch::kBFloat16);
  a.y = y.data_ptr();
  run_rows<NORM_BF16, STORE>(a);
  return y;
}

Tensor rows_norm_swiglu(Tensor x, Tensor norm, double eps, double add, Tensor w) {
  check_io(x, torch::kFloat32);
  CHK(w.size(0) % 2 == 0);
  auto a = rows_args(x, w, w.size(0) / 2);
  take_norm(a, norm, eps, add);
  auto y = rows_out(x, a.N, torch::kBFloat16);
  a.y = y.data_ptr();
  run_rows<NORM_F32, GATED_STORE>(a);
  return y;
}

Tensor rows_add_linear(Tensor x, Tensor w, Tensor res) {
  check_io(x, torch::kBFloat16);
  auto a = rows_args(x, w, w.size(0));
  const auto dt = io_type(res);
  CHK(res.numel() == (int64_t)a.m * a.N);
  a.res = res.data_ptr();
  auto y = torch::empty_like(res, res.options().dtype(dt == torch::kBFloat16 ? torch::kFloat32 : torch::kBFloat16));
  a.y = y.data_ptr();
  if (dt == torch::kBFloat16) run_rows<PLAIN_X, ADD_BF16>(a);
  else run_rows<PLAIN_X, ADD_F32>(a);
  return y;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rows_linear", &rows_linear);
  m.def("rows_norm_linear", &rows_norm_linear);
  m.def("rows_norm_swiglu", &rows_norm_swiglu);
  m.def("rows_add_linear", &rows_add_linear);
}
