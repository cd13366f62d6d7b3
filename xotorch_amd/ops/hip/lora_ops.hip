// The low-rank terms of adapted linears (bf16 rows; fp32 adapters A [r, K] and, turned so that
// a wave reads whole lines of it, B [r, N]; r <= 16):
//   sums   low [M, r] = t w^T and, of narrow rows c [M, r], t^T c
//   add    out += low w, where gemm_ops.hip does not add it inside the product
// (The reference has adapters as data only, train/data/lora.)
//
// What bounds them is t, read once, or out, read and written: library products of 8 features
// read a gradient once for either sum. us, library beside, 4096 tokens, rank 8: both sums of
// 28672 features 55 (126), of 4096 13 (41); the sum added to 28672 102 (132), to 14336 56 (72),
// to 4096 14 (19). Four layers of 4096 with 8 x 512 tokens, forward and back, 14300 (15500); 13700 with
// terms added inside the products.
// Here a block holds a strip of 256 columns of t and walks down its rows in steps of 64 through
// two LDS buffers; a step is multiplied along its rows and, read by transposing, along its
// columns. Sums of strips and of runs of rows are added up by another kernel, in order.
#include "mfma_tile.h"

struct SumArgs {
  const bf16_t* t;            // [M, N], N % 256 == 0
  const float* w;             // [r, N]
  const bf16_t* c;            // [16, Mp], zeros past r and M
  float *rows, *cols;         // [strips, M, rp], [chunks, N, rp]
  int M, N, r, rp, Mp, steps, per;  // steps of 64 rows, so many a block
};

// Eight numbers n .. of feature r of an adapter [rank, N], zeros past its rank
DEVINL void ld_adapter(const float* w, int n, int r, int rank, int N, float* o) {
  ld8(w + (size_t)min(r, rank - 1) * N + n, o);
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = r < rank ? o[j] : 0.f;
}

constexpr int STEP = 64 * 256;  // numbers of a buffer

// One row's pieces of a step, as ColFrags has its columns: 32 of the 256 each
struct StripFrags {
  bf16x8 f[8];
  unsigned at;
  DEVINL StripFrags(unsigned base, int row, int quad) { at = base + row * 512 + ((quad >> 1) ^ col_turn(row)) * 32 + (quad & 1) * 16; }
  template <int I>
  DEVINL void read(unsigned ring) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f[I]) : "v"((at ^ ((I & 3) << 6)) + ring), "i"((I >> 2) * 256));
  }
  DEVINL void landed() {
#pragma unroll
    for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(f[i]));
  }
};

template <bool ROWS, bool COLS>
__global__ __launch_bounds__(256, 2) void sums_kernel(SumArgs a) {
  extern __shared__ __attribute__((aligned(256))) bf16_t buf[];  // [2][64][256]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
  const int strips = a.N >> 8, strip = blockIdx.x % strips, chunk = blockIdx.x / strips, n0 = strip * 256;
  const int s0 = chunk * a.per, s1 = min(a.steps, s0 + a.per);
  auto send = [&](int s, int half) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = (wave * 8 + i) * 2 + (lane >> 5), piece = (lane & 31) ^ (col_turn(k) << 1);
      const bf16_t* from = a.t + (size_t)min(s * 64 + k, a.M - 1) * a.N + n0 + piece * 8;
      __builtin_amdgcn_global_load_lds((glb_void*)from, (lds_void*)(buf + half * STEP + (wave * 8 + i) * 512), 16, 0, 0);
    }
  };
  // narrow rows of a step
  bf16x8 now[2], next[2];
  auto narrow = [&](int s) {
#pragma unroll
    for (int h = 0; h < 2; ++h) next[h] = *(const bf16x8*)(a.c + (size_t)col * a.Mp + s * 64 + h * 32 + quad * 8);
  };
  if constexpr (COLS) narrow(s0);
  send(s0, 0);
  bf16x8 w[8];
  if constexpr (ROWS) {
    typedef __attribute__((ext_vector_type(8))) unsigned short ushort8_t;
    float v[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) ld_adapter(a.w, n0 + i * 32 + quad * 8, col, a.r, a.N, v[i]);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ushort8_t p;
#pragma unroll
      for (int j = 0; j < 8; ++j) p[j] = f2b(v[i][j]);
      w[i] = __builtin_bit_cast(bf16x8, p);
    }
  }
  const unsigned base = (unsigned)(size_t)(lds_void*)buf;
  const int mine = wave * 16 + col;  // a row of every step
  StripFrags x(base, mine, quad);
  ColFrags<4, 256> f(base, wave * 64, lane);
  floatx4 down[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) down[j] = (floatx4)(0.f);
  for (int s = s0; s < s1; ++s) {
    const int half = (s - s0) & 1;
    const unsigned ring = half * STEP * 2;
    if constexpr (COLS) now[0] = next[0], now[1] = next[1];
    if (s + 1 < s1) {
      if constexpr (COLS) narrow(s + 1);
      asm volatile("" ::: "memory");
      send(s + 1, half ^ 1);
      asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");  // all but what was just sent
      // (said here, as the compiler would wait for all loads where it copies these)
      if constexpr (COLS) asm volatile("" : "+v"(next[0]), "+v"(next[1]));
    } else {
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      const int left = a.M - s * 64;
      if (left < 64) {  // rows that are not there, and hold the last one, count as zeros
        for (int i = left * 32 + threadIdx.x; i < 64 * 32; i += 256) *(floatx4*)(buf + half * STEP + i * 8) = (floatx4)(0.f);
        __syncthreads();
      }
    }
    if constexpr (ROWS) {
      each<8>([&](auto i) { x.template read<decltype(i)::value>(ring); });
      reads_landed();
      x.landed();
      floatx4 sum = (floatx4)(0.f);
#pragma unroll
      for (int i = 0; i < 8; ++i) sum = mma(w[i], x.f[i], sum);
      const int m = s * 64 + mine;
      if (m < a.M && quad * 4 < a.rp) *(floatx4*)(a.rows + ((size_t)strip * a.M + m) * a.rp + quad * 4) = sum;
    }
    if constexpr (COLS) {
      each<2>([&](auto h) {
        constexpr int H = decltype(h)::value;
        each<8>([&](auto i) { f.template read<decltype(i)::value, H>(ring); });
        reads_landed();
        f.landed();
#pragma unroll
        for (int j = 0; j < 4; ++j) down[j] = mma(now[H], f[j], down[j]);
      });
    }
    asm volatile("s_barrier" ::: "memory");  // all have read it
  }
  if constexpr (COLS)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (quad * 4 < a.rp) *(floatx4*)(a.cols + ((size_t)chunk * a.N + n0 + wave * 64 + j * 16 + col) * a.rp + quad * 4) = down[j];
}

struct MergeArgs {
  const float *rows, *cols;  // as above
  float *low, *out;          // [M, rp]; [N, r], or [r, N] if turned
  bf16_t* lowt;              // [16, Mp]
  int M, N, r, rp, Mp, strips, chunks, row_blocks;
  float row_scale, col_scale;
  bool turned;
};

// Four sums of 32 places a block, eight threads each
__global__ __launch_bounds__(256) void merge_kernel(MergeArgs a) {
  __shared__ floatx4 part[8][32];
  const bool down = (int)blockIdx.x >= a.row_blocks;
  const int lane = threadIdx.x & 31, nth = threadIdx.x >> 5, at = (blockIdx.x - (down ? a.row_blocks : 0)) * 32 + lane;
  const int quads = down ? a.rp / 4 : 4, i = at / quads, q = at % quads, most = down ? a.N : a.M, parts = down ? a.chunks : a.strips;
  floatx4 sum = (floatx4)(0.f);
  if (i < most && q * 4 < a.rp) {
    const float* from = (down ? a.cols : a.rows) + (size_t)i * a.rp + q * 4;
#pragma unroll 4
    for (int p = nth; p < parts; p += 8) sum += *(const floatx4*)(from + (size_t)p * most * a.rp);
  }
  part[nth][lane] = sum;
  __syncthreads();
  if (nth) return;
#pragma unroll
  for (int p = 1; p < 8; ++p) sum += part[p][lane];
  sum *= down ? a.col_scale : a.row_scale;
  // what fills a rank up are products with zeros, so no numbers where t has an infinity
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (q * 4 + e >= a.r) sum[e] = 0.f;
  if (down) {
    if (i >= most) return;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (q * 4 + e < a.r) a.out[a.turned ? (size_t)(q * 4 + e) * a.N + i : (size_t)i * a.r + q * 4 + e] = sum[e];
  } else {
    if (i < most && q * 4 < a.rp) *(floatx4*)(a.low + (size_t)i * a.rp + q * 4) = sum;
    if (i < a.Mp)
#pragma unroll
      for (int e = 0; e < 4; ++e) a.lowt[(size_t)(q * 4 + e) * a.Mp + i] = f2b(sum[e]);
  }
}

// out [M, N] += scale low w of an adapter [rank, N]: a lane has eight columns of w, and walks
// down `group` rows
template <int RP>
__global__ __launch_bounds__(256) void add_kernel(bf16_t* out, const float* __restrict__ low, const float* __restrict__ w, int M, int N,
                                                  int rank, float scale, int group) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int strips = (N + 511) / 512, n = blockIdx.x % strips * 512 + lane * 8;
  const int m0 = (blockIdx.x / strips * 4 + wave) * group, m1 = min(M, m0 + group);
  if (n >= N || m0 >= M) return;
  float by[RP][8];
#pragma unroll
  for (int r = 0; r < RP; ++r) ld_adapter(w, n, r, rank, N, by[r]);
#pragma unroll
  for (int r = 0; r < RP; ++r)
#pragma unroll
    for (int j = 0; j < 8; ++j) by[r][j] *= scale;
  typedef __attribute__((ext_vector_type(8))) unsigned short ushort8_t;
  constexpr int AT_ONCE = 8;
  for (int m = m0; m < m1; m += AT_ONCE) {
    ushort8_t v[AT_ONCE];
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i) v[i] = *(const ushort8_t*)(out + (size_t)min(m + i, m1 - 1) * N + n);
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i) {
      if (m + i >= m1) break;
      const float* l = low + (size_t)(m + i) * RP;
      float o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = __uint_as_float((unsigned)v[i][j] << 16);
#pragma unroll
      for (int r = 0; r < RP; ++r)
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] += l[r] * by[r][j];
      ushort8_t y;
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = f2b(o[j]);
      *(ushort8_t*)(out + (size_t)(m + i) * N + n) = y;
    }
  }
}

// ===========================================================================
// host side
// ===========================================================================
static int padded(int64_t rank) { return rank <= 4 ? 4 : rank <= 8 ? 8 : 16; }

static void check_rows(const Tensor& t) {
  check_io(t, torch::kBFloat16);
  CHK(t.dim() == 2 && t.size(0) >= 1 && t.size(0) <= 1 << 22 && t.size(1) >= 256 && t.size(1) <= 1 << 22 && t.size(1) % 256 == 0);
  CHK(((size_t)t.data_ptr() & 15) == 0);
}
static void check_adapter(const Tensor& w, int64_t n, int64_t rank) {
  check_io(w, torch::kFloat32);
  CHK(w.dim() == 2 && w.size(1) == n && w.size(0) == rank && rank >= 1 && rank <= 16 && ((size_t)w.data_ptr() & 15) == 0);
}

// (low [M, rp], the same as bf16 columns [16, Mp]) = scale t w^T where w [rank, N] is given; t^T c (c as such
// columns) times col_scale, [N, rank] or [rank, N], where c is
std::vector<Tensor> low_rank_sums(Tensor t, OptT w, double scale, OptT c, int64_t rank, double col_scale, bool col_turned) {
  check_rows(t);
  CHK((w || c) && rank >= 1 && rank <= 16);
  SumArgs a{};
  a.t = P<bf16_t>(t);
  a.M = (int)t.size(0);
  a.N = (int)t.size(1);
  a.r = (int)rank;
  a.rp = padded(rank);
  a.steps = (a.M + 63) / 64;
  a.Mp = a.steps * 64;
  const int strips = a.N / 256, chunks = std::min(a.steps, std::max(1, 512 / strips));
  a.per = (a.steps + chunks - 1) / chunks;
  MergeArgs m{};
  m.M = a.M, m.N = a.N, m.r = a.r, m.rp = a.rp, m.Mp = a.Mp, m.strips = strips, m.chunks = (a.steps + a.per - 1) / a.per;
  m.row_scale = (float)scale, m.col_scale = (float)col_scale, m.turned = col_turned;
  std::vector<Tensor> found;
  Tensor rows, cols;
  int blocks = 0;
  if (w) {
    check_adapter(*w, a.N, rank);
    a.w = P<float>(*w);
    rows = f32(t, {strips, a.M, a.rp});
    m.rows = a.rows = rows.data_ptr<float>();
    found.push_back(f32(t, {a.M, a.rp}));
    found.push_back(torch::empty({16, a.Mp}, t.options()));
    m.low = found[0].data_ptr<float>();
    m.lowt = M<bf16_t>(found[1]);
    blocks = m.row_blocks = a.Mp / 8;  // 32 of [Mp, 4]
  }
  if (c) {
    check_io(*c, torch::kBFloat16);
    CHK(c->dim() == 2 && c->size(0) == 16 && c->size(1) == a.Mp && ((size_t)c->data_ptr() & 15) == 0);
    a.c = P<bf16_t>(*c);
    cols = f32(t, {m.chunks, a.N, a.rp});
    m.cols = a.cols = cols.data_ptr<float>();
    found.push_back(col_turned ? f32(t, {rank, a.N}) : f32(t, {a.N, rank}));
    m.out = found.back().data_ptr<float>();
    blocks += a.N * (a.rp / 4) / 32;
  }
  auto run = [&](auto kernel) {
    constexpr int lds = 2 * STEP * (int)sizeof(bf16_t);
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    TORCH_CHECK(e == hipSuccess, "no LDS for low-rank sums");
    hipLaunchKernelGGL(kernel, dim3(strips * m.chunks), dim3(256), lds, cur_stream(), a);
  };
  if (w && c) run(sums_kernel<true, true>);
  else if (w) run(sums_kernel<true, false>);
  else run(sums_kernel<false, true>);
  hipLaunchKernelGGL(merge_kernel, dim3(blocks), dim3(256), 0, cur_stream(), m);
  return found;
}

// out [M, N] += scale low w of an adapter [rank, N]
void low_rank_add(Tensor out, Tensor low, Tensor w, double scale) {
  check_rows(out);
  check_io(low, torch::kFloat32);
  const int64_t rank = w.size(0);
  check_adapter(w, out.size(1), rank);
  CHK(low.dim() == 2 && low.size(0) == out.size(0) && low.size(1) == padded(rank));
  const int rows = (int)out.size(0), N = (int)out.size(1), strips = (N + 511) / 512;
  // rows that share what a wave has of w, as long as eight waves a CU are left
  const int group = (int)std::min<int64_t>(64, std::max<int64_t>(8, (int64_t)rows * strips / 2048 / 8 * 8));
  const dim3 grid((unsigned)((rows + group * 4 - 1) / (group * 4) * strips));
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, cur_stream(), M<bf16_t>(out), low.data_ptr<float>(), P<float>(w), rows, N, (int)rank,
                       (float)scale, group);
  };
  if (padded(rank) == 4) run(add_kernel<4>);
  else if (padded(rank) == 8) run(add_kernel<8>);
  else run(add_kernel<16>);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("sums", &low_rank_sums, "t w^T of t [M, N] and an adapter [rank, N], t^T c");
  m.def("add", &low_rank_add, "out += scale low w");
}
