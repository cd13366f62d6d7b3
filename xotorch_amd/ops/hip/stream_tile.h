// Products of few rows of x, which the weights' way from memory bounds: a block's weight rows
// and rows of x go through a ring of LDS buffers in steps of 64 along k, by direct loads: rows of 128
// bytes, so whole lines, the 16-byte pieces of row r permuted by r & 7 in the global
// address, which spreads fragment reads over the banks.
#pragma once
#include "mfma_tile.h"

// R fragments from a on and C from b on, 16 rows (2 KB) apart; waits for them
template <int R, int C>
DEVINL void read_frags(unsigned a, unsigned b, bf16x8* r, bf16x8* c) {
#define RD(D, A, O) "ds_read_b128 %" #D ", %" #A " offset:" #O "\n\t"
#define DONE "s_waitcnt lgkmcnt(0)"
  if constexpr (R == 1 && C == 1)
    asm volatile(RD(0, 2, 0) RD(1, 3, 0) DONE : "=&v"(r[0]), "=&v"(c[0]) : "v"(a), "v"(b));
  else if constexpr (R == 1 && C == 2)
    asm volatile(RD(0, 3, 0) RD(1, 4, 0) RD(2, 4, 2048) DONE : "=&v"(r[0]), "=&v"(c[0]), "=&v"(c[1]) : "v"(a), "v"(b));
  else if constexpr (R == 1 && C == 4)
    asm volatile(RD(0, 5, 0) RD(1, 6, 0) RD(2, 6, 2048) RD(3, 6, 4096) RD(4, 6, 6144) DONE
                 : "=&v"(r[0]), "=&v"(c[0]), "=&v"(c[1]), "=&v"(c[2]), "=&v"(c[3]) : "v"(a), "v"(b));
  else if constexpr (R == 2 && C == 1)
    asm volatile(RD(0, 3, 0) RD(1, 3, 2048) RD(2, 4, 0) DONE : "=&v"(r[0]), "=&v"(r[1]), "=&v"(c[0]) : "v"(a), "v"(b));
  else if constexpr (R == 2 && C == 2)
    asm volatile(RD(0, 4, 0) RD(1, 4, 2048) RD(2, 5, 0) RD(3, 5, 2048) DONE
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(c[0]), "=&v"(c[1]) : "v"(a), "v"(b));
  else {
    static_assert(R == 4 && C == 2, "");
    asm volatile(RD(0, 6, 0) RD(1, 6, 2048) RD(2, 6, 4096) RD(3, 6, 6144) RD(4, 7, 0) RD(5, 7, 2048) DONE
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(c[0]), "=&v"(c[1]) : "v"(a), "v"(b));
  }
#undef RD
#undef DONE
}

template <int BN_, int BM_, int BUFS_, int WAVES_ = 4>
struct TileShape {
  static constexpr int BN = BN_, BM = BM_, BUFS = BUFS_, ROWS = BN + BM, BUF = ROWS * 64;  // elements of a buffer
  static constexpr int WAVES = WAVES_;
  static constexpr int WL = BN / 8 / WAVES, XL = BM >= 32 ? BM / 32 : 1;  // loads of a wave and stage; of x by four
  static constexpr int LDS = BUFS * BUF * 2;
  // waves along x: the weight rows are split over all of them for few rows of x, or more than four
  static constexpr int WX = BM >= 64 && WAVES == 4 ? 2 : 1, R = BN * WX / WAVES / 16, C = BM / WX / 16;
  // a wave's first weight row and row of x
  static DEVINL int wr(int wave) { return wave / WX * (R * 16); }
  static DEVINL int wx(int wave) { return wave % WX * (C * 16); }
};

// acc = the sum over `len` steps of 64. wsrc, xsrc: where this lane's pieces of 16 bytes begin: weights in loads
// of 8 rows, WL a wave, row wave * WL * 8 + i * 8 + lane / 8 of the tile; x by four waves, XL a wave, of 8 rows (16
// rows of x: of 4 rows), which further waves load again; piece (lane & 7) ^ (row & 7). turn: the step that
// comes first.
template <typename Sh>
DEVINL void stream_walk(floatx4 (&acc)[Sh::R][Sh::C], bf16_t* buf, const bf16_t* (&wsrc)[Sh::WL], const bf16_t* (&xsrc)[Sh::XL],
                        int len, int turn, int wave, int lane) {
  constexpr int BN = Sh::BN, BM = Sh::BM, BUFS = Sh::BUFS, R = Sh::R, C = Sh::C, LOADS = Sh::WL + Sh::XL;
  const int col = lane & 15, quad = lane >> 4;
  auto stage = [&](int s) {
    bf16_t* dst = buf + (s % BUFS) * Sh::BUF;
    const int k = (s + turn < len ? s + turn : s + turn - len) * 64;
#pragma unroll
    for (int i = 0; i < Sh::WL; ++i)
      __builtin_amdgcn_global_load_lds((glb_void*)(wsrc[i] + k), (lds_void*)(dst + (wave * Sh::WL + i) * 512), 16, 0, 2);
#pragma unroll
    for (int i = 0; i < Sh::XL; ++i) {
      bf16_t* to = dst + BN * 64 + (wave & 3) * (BM >= 32 ? Sh::XL * 512 : 256) + i * 512;
      if (BM >= 32 || lane < 32)
        __builtin_amdgcn_global_load_lds((glb_void*)(xsrc[i] + k), (lds_void*)to, 16, 0, 0);
    }
  };
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < C; ++j) acc[i][j] = (floatx4)(0.f);
#pragma unroll
  for (int i = 0; i < BUFS - 1; ++i)
    if (i < len) stage(i);
  // this lane's first fragments, as LDS byte addresses within a buffer
  const unsigned base = (unsigned)(size_t)(lds_void*)buf;
  const unsigned wl = base + (Sh::wr(wave) + col) * 128, xl = base + (BN + Sh::wx(wave) + col) * 128;
  const unsigned place[2] = {(unsigned)((quad ^ (col & 7)) * 16), (unsigned)(((4 + quad) ^ (col & 7)) * 16)};
  for (int s = 0; s < len; ++s) {
    // this step is in LDS, up to BUFS - 2 later ones are on their way; the buffer of
    // the step before is free
    const int left = min(BUFS - 2, len - 1 - s);
    if (left >= 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(2 * LOADS) : "memory");
    else if (left == 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    if (s + BUFS - 1 < len) stage(s + BUFS - 1);
    const unsigned at = (unsigned)(s % BUFS) * (Sh::BUF * 2);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8 wf[R], xf[C];
      read_frags<R, C>(wl + at + place[h], xl + at + place[h], wf, xf);
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < C; ++j) acc[i][j] = mma(wf[i], xf[j], acc[i][j]);
    }
  }
}
