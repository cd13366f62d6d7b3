// Products of weight rows and rows of x whose tiles are walked in steps of 64 along k
// through two rings of LDS buffers, one for either operand: what the kernels share that
// are bound by the matrix cores.
//
// Eight waves, two a SIMD. LDS rows hold 8 pieces of 16 bytes, piece p of row r at place
// p ^ (r & 7): loads go straight to LDS lane by lane, so the permutation sits in the global
// address, and fragment reads spread over the banks. A wave multiplies one half of a step
// (32 of k) while it reads the fragments of the next half, so that matrix cores do not wait
// for LDS: a step's last reads are over in the middle of it, where its one barrier lies,
// and the loads that take its buffers are sent behind that. Weights come from farther than
// x does and are sent further ahead: of 256 x 256, three buffers of weights and two of x
// are the 160 KB that a CU has.
//
// [4096, 4096] x [28672, 4096]^T, 256 x 256 a block: 1.41 PFLOP/s (two buffers of both 1.35;
// without any loads 1.74; matrix instructions alone 2.15). Four waves of 128 x 128 read
// less of LDS and reach 1.30. Which blocks share a die's L2 counts as much: 1.32 where 32
// neighbours read 32 weight tiles and one of x, 1.41 to 1.43 in patches of 4 by 8.
#pragma once
#include "common.h"

#include <utility>

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void glb_void;

// f(0), f(1) .. f(N - 1), each with its number as a constant
template <typename F, int... I>
DEVINL void each_of(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>()), ...); }
template <int N, typename F>
DEVINL void each(F&& f) { each_of(f, std::make_integer_sequence<int, N>()); }

// BN weight rows and BM rows of x, WN waves along the weights; WB and XB buffers. A wave
// has R x C tiles of 16.
template <int BN, int BM, int WN, int WB_, int XB_>
struct MfmaTile {
  static constexpr int WAVES = 8, R = BN / WN / 16, C = BM * WN / WAVES / 16;
  static constexpr int WB = WB_, XB = XB_, WL = (BN / 8 + WAVES - 1) / WAVES, XL = BM / 8 / WAVES;  // 8 rows a load and wave
  static constexpr int WBYTES = BN * 128, XBYTES = BM * 128, XAT = WB * WBYTES, LDS = XAT + XB * XBYTES;
  static_assert(BN % (WN * 16) == 0 && BM * WN % (WAVES * 16) == 0 && BM % 64 == 0 && LDS <= 160 * 1024 && WB >= XB && XB >= 2, "");
};

// One operand's fragments of 32 of k, N tiles of 16 rows, and where a lane reads them. By
// hand: the compiler would make every read wait for all pending loads to LDS. What is read
// is used, after `landed`.
//
// Rows: k lies along a row, as above.
template <int N>
struct RowFrags {
  static constexpr int COUNT = N;  // reads
  bf16x8 f[N];
  unsigned at[2];  // of either half of a step
  // the fragments from row `row` on of buffers at byte `base`
  DEVINL RowFrags(unsigned base, int row, int lane) {
    const int col = lane & 15, quad = lane >> 4;
#pragma unroll
    for (int h = 0; h < 2; ++h) at[h] = base + (row + col) * 128 + (((h * 4 + quad) ^ (col & 7)) * 16);
  }
  template <int I, int H>
  DEVINL void read(unsigned ring) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f[I]) : "v"(at[H] + ring), "i"(I * 2048));
  }
  DEVINL void landed() {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
  }
  DEVINL bf16x8 operator[](int i) const { return f[i]; }
  DEVINL void clear(int, int, int) {}
};

// Columns: a step is 64 rows of F numbers, k along the rows. Transposing reads give a lane
// four k of its column; the chunks of 32 bytes of row k are permuted by g(k) of 0 .. 7, so
// that the four rows of a read, and the eight of two, lie in different banks.
DEVINL int col_turn(int k) { return (k & 3) | (k >> 1 & 4); }
template <int N, int F>
struct ColFrags {
  static constexpr int COUNT = 2 * N;
  typedef __attribute__((ext_vector_type(4))) __bf16 half_t;
  half_t lo[N], hi[N];
  unsigned at;  // of the first tile; that of tile i differs in bits 5 to 7
  DEVINL ColFrags(unsigned base, int col, int lane) {
    const int k = (lane >> 4) * 8 + ((lane & 15) >> 2);
    at = base + k * (F * 2) + ((col >> 4) ^ col_turn(k)) * 32 + (lane & 3) * 8;
  }
  template <int I, int H>
  DEVINL void read(unsigned ring) {
    const unsigned a = (at ^ ((I / 2) << 5)) + ring;
    if constexpr (I % 2 == 0) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo[I / 2]) : "v"(a), "i"(H * 64 * F));
    else asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi[I / 2]) : "v"(a), "i"(H * 64 * F + 8 * F));
  }
  DEVINL void landed() {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      asm volatile("" : "+v"(lo[i]));
      asm volatile("" : "+v"(hi[i]));
    }
  }
  DEVINL bf16x8 operator[](int i) const { return __builtin_shufflevector(lo[i], hi[i], 0, 1, 2, 3, 4, 5, 6, 7); }
  // zeros for the step's first `skip` k, of half h
  DEVINL void clear(int skip, int h, int lane) {
    typedef __attribute__((ext_vector_type(4))) short short4_t;
    const int n = skip - h * 32 - (lane >> 4) * 8;  // of this lane's eight
    short4_t a, b;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a[e] = e < n ? 0 : -1;
      b[e] = e + 4 < n ? 0 : -1;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      lo[i] = __builtin_bit_cast(half_t, (short4_t)(__builtin_bit_cast(short4_t, lo[i]) & a));
      hi[i] = __builtin_bit_cast(half_t, (short4_t)(__builtin_bit_cast(short4_t, hi[i]) & b));
    }
  }
};
DEVINL void reads_landed() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// acc += over `steps` steps (one at least). loadw(i, s, at): this wave's load i of WL of
// step s, to byte `at` of LDS, loadx the same; w, x: this lane's fragments (RowFrags or
// ColFrags), which read from the first buffers on; skip: k of the last step that do not count.
template <typename T, int R, int C, typename W, typename X, typename LoadW, typename LoadX>
DEVINL void walk(floatx4 (&acc)[R][C], W w, X x, int steps, LoadW loadw, LoadX loadx, int skip = 0) {
  constexpr int WB = T::WB, XB = T::XB, WL = T::WL, XL = T::XL, AHEAD = WB - XB;
  W wa = w, wb = w;
  X xa = x, xb = x;
  // read number k of a half: x first
  auto read = [&](auto number, auto half, W& fw, X& fx, unsigned wring, unsigned xring) {
    constexpr int k = decltype(number)::value, h = decltype(half)::value;
    if constexpr (k < X::COUNT) fx.template read<k, h>(xring);
    else if constexpr (k < X::COUNT + W::COUNT) fw.template read<k - X::COUNT, h>(wring);
  };
  const std::integral_constant<int, 0> first;
  const std::integral_constant<int, 1> second;
  auto send_w = [&](int s, unsigned at) { each<WL>([&](auto i) { loadw(i, s, at); }); };
  auto send_x = [&](int s, unsigned at) { each<XL>([&](auto i) { loadx(i, s, at); }); };
  // the order of the loads is that of the loop: x of a step, then weights of AHEAD steps later
#pragma unroll
  for (int s = 0; s < AHEAD; ++s)
    if (s < steps) send_w(s, s * T::WBYTES);
#pragma unroll
  for (int s = 0; s < XB; ++s) {
    if (s < steps) send_x(s, T::XAT + s * T::XBYTES);
    if (s + AHEAD < steps) send_w(s + AHEAD, (s + AHEAD) * T::WBYTES);
  }
  // loads that may still be on their way when the next step's have to be there
  constexpr int LATER = (AHEAD ? WL : 0) + (XB - 2) * (XL + WL);
  if (steps >= WB) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(LATER + XL + WL) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  constexpr int READS = X::COUNT + W::COUNT;
  each<READS>([&](auto k) { read(k, first, wa, xa, 0, 0); });
  // behind a row of products: all reads in the first half of them, all loads in as many rows
  constexpr int PER = (2 * READS + R - 1) / R, LPER = (WL + XL + R - 1) / R;
  unsigned wu = 0, xu = 0;  // this step's buffers
  // more: another step follows; fill: all loads go on
  auto step = [&](int s, auto more, auto fill) {
    reads_landed();
    xa.landed();
    wa.landed();
    if (!decltype(more)::value && skip > 0) {
      xa.clear(skip, 0, threadIdx.x & 63);
      wa.clear(skip, 0, threadIdx.x & 63);
    }
    each<R>([&](auto row) {
      constexpr int i = decltype(row)::value;
#pragma unroll
      for (int j = 0; j < C; ++j) acc[i][j] = mma(wa[i], xa[j], acc[i][j]);
      each<PER>([&](auto n) { read(std::integral_constant<int, i * PER + decltype(n)::value>(), second, wb, xb, wu, xu); });
      __builtin_amdgcn_sched_barrier(0);
    });
    reads_landed();
    xb.landed();
    wb.landed();
    if (!decltype(more)::value && skip > 0) {
      xb.clear(skip, 1, threadIdx.x & 63);
      wb.clear(skip, 1, threadIdx.x & 63);
    }
    const unsigned w0 = wu, x0 = T::XAT + xu;
    if constexpr (decltype(more)::value) {
      // all waves have read this step, and the next one is there
      if constexpr (decltype(fill)::value) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(LATER) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      wu = wu == (WB - 1) * T::WBYTES ? 0 : wu + T::WBYTES;
      xu = xu == (XB - 1) * T::XBYTES ? 0 : xu + T::XBYTES;
      if (!decltype(fill)::value && s + XB < steps) send_x(s + XB, x0);
    }
    each<R>([&](auto row) {
      constexpr int i = decltype(row)::value;
#pragma unroll
      for (int j = 0; j < C; ++j) acc[i][j] = mma(wb[i], xb[j], acc[i][j]);
      if constexpr (decltype(more)::value)
        each<PER>([&](auto n) { read(std::integral_constant<int, i * PER + decltype(n)::value>(), first, wa, xa, wu, xu); });
      if constexpr (decltype(fill)::value)
        each<LPER>([&](auto n) {
          constexpr int k = i * LPER + decltype(n)::value;
          if constexpr (k < XL) loadx(std::integral_constant<int, k>(), s + XB, x0);
          else if constexpr (k < XL + WL) loadw(std::integral_constant<int, k - XL>(), s + WB, w0);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  const std::true_type yes;
  const std::false_type no;
  int s = 0;
  for (; s + WB < steps; ++s) step(s, yes, yes);
  for (; s + 1 < steps; ++s) step(s, yes, no);
  step(s, no, no);
}
