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

template <int R, int C> struct Frags { bf16x8 w[R], x[C]; };

// The fragments at bytes w and x of LDS, 16 rows apart: x first, then w; number I of them
template <int I, int R, int C>
DEVINL void read_frag(Frags<R, C>& f, unsigned w, unsigned x) {
  // by hand: the compiler would make every read wait for all pending loads to LDS. What is
  // read here is used, after `landed`
  if constexpr (I < C) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.x[I]) : "v"(x), "i"(I * 2048));
  else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.w[I - C]) : "v"(w), "i"((I - C) * 2048));
}
template <int R, int C>
DEVINL void landed(Frags<R, C>& f) {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < C; ++i) asm volatile("" : "+v"(f.x[i]));
#pragma unroll
  for (int i = 0; i < R; ++i) asm volatile("" : "+v"(f.w[i]));
}

// acc += over `steps` steps (one at least). loadw(i, s, at): this wave's load i of WL of
// step s, to byte `at` of LDS, loadx the same; wl, xl: this lane's first fragments within
// the first buffers; place: where a half's pieces lie.
template <typename T, int R, int C, typename LoadW, typename LoadX>
DEVINL void walk(floatx4 (&acc)[R][C], unsigned wl, unsigned xl, const unsigned (&place)[2], int steps, LoadW loadw, LoadX loadx) {
  constexpr int WB = T::WB, XB = T::XB, WL = T::WL, XL = T::XL, AHEAD = WB - XB;
  Frags<R, C> a, b;
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
  each<R + C>([&](auto i) { read_frag<decltype(i)::value>(a, wl + place[0], xl + place[0]); });
  // behind a row of products: all reads in the first half of them, all loads in as many rows
  constexpr int PER = (2 * (R + C) + R - 1) / R, LPER = (WL + XL + R - 1) / R;
  unsigned wu = 0, xu = 0;  // this step's buffers
  // more: another step follows; fill: all loads go on
  auto step = [&](int s, auto more, auto fill) {
    landed(a);
    each<R>([&](auto row) {
      constexpr int i = decltype(row)::value;
#pragma unroll
      for (int j = 0; j < C; ++j) acc[i][j] = mma(a.w[i], a.x[j], acc[i][j]);
      each<PER>([&](auto n) {
        constexpr int k = i * PER + decltype(n)::value;
        if constexpr (k < R + C) read_frag<k>(b, wl + wu + place[1], xl + xu + place[1]);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    landed(b);
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
      for (int j = 0; j < C; ++j) acc[i][j] = mma(b.w[i], b.x[j], acc[i][j]);
      if constexpr (decltype(more)::value)
        each<PER>([&](auto n) {
          constexpr int k = i * PER + decltype(n)::value;
          if constexpr (k < R + C) read_frag<k>(a, wl + wu + place[0], xl + xu + place[0]);
        });
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
