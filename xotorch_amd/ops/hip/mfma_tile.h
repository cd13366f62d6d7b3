// Products of weight rows and rows of x whose tiles are walked in steps of 64 along k
// through two rings of LDS buffers, one for either operand: what the kernels share that
// are bound by the matrix cores.
//
// LDS rows hold 8 pieces of 16 bytes, piece p of row r at place p ^ (r & 7): loads go straight
// to LDS lane by lane, so the permutation sits in the global address, and fragment reads spread
// over the banks. A wave multiplies one half of a step (32 of k) while it reads the fragments
// of the next half, so that matrix cores do not wait for LDS: a step's last reads are over in
// the middle of it, where its one barrier lies, and the loads that take its buffers are sent
// one by one over the step's length behind that. Weights come from farther than x does and
// are sent further ahead: of 256 x 256, three buffers of weights and two of x are the 160 KB
// that a CU has.
//
// Four waves, one a SIMD, or eight: the larger a wave's part of a tile, the fewer fragments it
// reads for a product, but two waves a SIMD begin and end a block faster. 256 blocks of 256 x
// 256, of 512, 1024 and 4096 of k, us, four first: 22.1, 21.0; 33.7, 32.4; 100, 99; of 128 x
// 256 14.4, 13.7; 20.5, 19.6; 58.1, 56.9; where both operands are columns of 256 x 256 25.0,
// 21.9; 37.0, 33.1; 109, 104. So where rows of x fill their tiles eight gain 1 to 5%, more of short
// sums; but only four make tiles of any multiple of 32 rows of x, eight of 64. Experts and gates of
// prompts, whose rows are shared out, take four: 300 and 600 rows by [28672, 4096] 70 and 137, 87 and
// 140; 600 by [16384, 8192] 132, 152; by [16384, 2048] 38.6, 42.0; 8 experts of 4096 x 14336, 250 rows
// each, 467 and 235, 478 and 244; from 1000 rows of 1024 and more on 0.97 to 1.02 (1500 wide 1.04 to 1.09).
// Rows of less than 1024 lose by it: 3000 by [9728, 896] 53.0, 50.1 (600 16.7, 14.7; 2000 37.6, 41.1), by
// [9728, 256] 25.5, 23.2; 16 experts of 1024 x 512, 250 rows each, 20.4, 18.8. One set of tiles serves
// all, as two would double the largest kernels.
//
// What bounds large tiles is power: [6144, 4096] x [28672, 4096]^T, 256 x 256 a block, takes
// 2390 to 2500 cycles a step of the 2048 that its matrix instructions need, at 1.8 GHz of 2.4
// (matrix instructions alone run at 2.1). PFLOP/s, four waves, and as it was with eight whose
// loads took addresses in registers and whose results went out from them: 256 x 256 1.40
// (1.34), 256 x 192 1.33 (1.26), one round of 160 x 256 1.11 (0.95). Which blocks share a die's
// L2 counts as much: 1.32 where 32 neighbours read 32 weight tiles and one of x, 1.41 to 1.43
// in patches of 4 by 8.
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
template <int BN, int BM, int WN, int WB_, int XB_, int WAVES_ = 4>
struct MfmaTile {
  static constexpr int WAVES = WAVES_, THREADS = WAVES * 64, R = BN / WN / 16, C = BM * WN / WAVES / 16;
  static constexpr int WB = WB_, XB = XB_, WL = BN / 8 / WAVES, XL = BM / 8 / WAVES;  // 8 rows a load and wave
  static constexpr int WBYTES = BN * 128, XBYTES = BM * 128, XAT = WB * WBYTES, LDS = XAT + XB * XBYTES;
  static_assert(BN % (WN * 16) == 0 && BM * WN % (WAVES * 16) == 0 && BN % (8 * WAVES) == 0 && BM % (8 * WAVES) == 0 && LDS <= 160 * 1024, "");
  static_assert(WB >= XB && XB >= 2 && C >= 2 && R * C >= 8, "");
};

// Where one step's loads come from, up to 4 GB from `base` on: a lane's offset stays in a
// register and a step's is a scalar, so that a load takes no address of its own to compute
// (64-bit addresses in registers cost 3% of a product). A step past the last is a buffer
// without records, of which nothing is read; its offset is 0, as the hardware asks whether a
// lane's offset lies past the records less the scalar, which would wrap round.
struct StepSource {
  const void* base;
  unsigned at;  // bytes
  int mask;     // -1; past the last step 0
  DEVINL StepSource(const void* base_, unsigned at_, int left) : base(base_), mask(there(left)) { at = at_ & mask; }
  // -1 where steps are left, else 0. By hand: of a comparison the compiler makes a vector, takes
  // the buffer for another one in every lane, and loops over the lanes around each load.
  static DEVINL int there(int left) {
    int mask = 0;
#ifdef __HIP_DEVICE_COMPILE__
    asm("s_ashr_i32 %0, %1, 31" : "=s"(mask) : "s"(-left) : "scc");
#endif
    return mask;
  }
  // 16 bytes a lane to LDS. AUX 2: of lines that nobody reads again
  template <int AUX = 0>
  DEVINL void load(unsigned lane_at, void* to) const {
#ifdef __HIP_DEVICE_COMPILE__  // the host's compiler does not know the type
    const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, mask, 0x20000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_void*)to, 16, lane_at, at, 0, AUX);
#endif
  }
};

// One operand's fragments of 32 of k, N tiles of 16 rows, and where a lane reads them. By
// hand: the compiler would make every read wait for all pending loads to LDS. What is read
// is used after `landed`: fragment i as [i] by instructions that the compiler knows, as f[i],
// behind `whole` too, by those that it does not (`mul`).
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
  DEVINL void whole() { landed(); }
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
  bf16x8 f[N];
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
  // both halves where they are multiplied, before `written`
  DEVINL void whole() {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      f[i] = (*this)[i];
      asm volatile("" : "+v"(f[i]));
    }
  }
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

// Sums stay in the accumulation registers they are in. By hand: the compiler gives a wave's
// 256 of them new places and moves them there, 20 moves and 16 waits a step (2780 cycles of
// 256 x 256 in four waves, 2500 so). A sum's next is at least 8 of them later, and none follows closely
// on something else that writes what it reads (`written`).
DEVINL void mul(floatx4& sum, const bf16x8& a, const bf16x8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(sum) : "v"(a), "v"(b));
}
// The same of a step's last product. Behind the last step (more: steps that are left) it waits until
// all sums are written, in the same block: the compiler, which knows nothing of them, may move sums
// anywhere behind the loop, and did. That lies behind the kernel's end, as steps before the last
// would jump over it: 1% of gates of prompts, 0.4% so (0.3 to 0.6% of all products).
DEVINL void mul_last(floatx4& sum, const bf16x8& a, const bf16x8& b, int more) {
#ifdef __HIP_DEVICE_COMPILE__
#define MUL "v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
  asm volatile("s_cmp_lg_u32 %3, 0\n\ts_cbranch_scc0 .Llast%=\n\t" MUL "\n.Lgone%=:\n\t"
               ".subsection 1\n.Llast%=:\n\t" MUL "s_nop 15\n\ts_nop 7\n\ts_branch .Lgone%=\n\t.previous"
               : "+a"(sum) : "v"(a), "v"(b), "s"(__builtin_amdgcn_readfirstlane(more)) : "scc");
#undef MUL
#endif
}
// Two cycles between a write of registers and the instructions above
DEVINL void written() { asm volatile("s_nop 1" ::: "memory"); }

// acc = the sum over `steps` steps (one at least). stepw(s): where step s of the weights comes
// from, loadw(i, that, at): this wave's load i of WL of it, to byte `at` of LDS; stepx and
// loadx the same; steps past the last count as loads but have nothing to bring, so that one
// loop does for all steps, and sums are never moved. w, x: this lane's fragments (RowFrags or
// ColFrags), which read from the first buffers on; skip: k of the last step that do not count.
// All of LDS is free when it returns.
template <typename T, int R, int C, typename W, typename X, typename StepW, typename LoadW, typename StepX, typename LoadX>
DEVINL void walk(floatx4 (&acc)[R][C], W w, X x, int steps, StepW stepw, LoadW loadw, StepX stepx, LoadX loadx, int skip = 0) {
  constexpr int WB = T::WB, XB = T::XB, WL = T::WL, XL = T::XL, AHEAD = WB - XB, ALL = WL + XL;
  // loads behind a row of products, and how many of a step's are sent before the next begins
  constexpr int LPER = (ALL + 2 * R - 1) / (2 * R), NOW = ALL < LPER * R ? ALL : LPER * R;
  // reads behind either half of a row: all of them in the first half of the rows
  constexpr int READS = X::COUNT + W::COUNT, PER = ((READS + (R + 1) / 2 - 1) / ((R + 1) / 2) + 1) / 2;
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < C; ++j) acc[i][j] = (floatx4)(0.f);
  W wa = w, wb = w;
  X xa = x, xb = x;
  // read number k of a half: x first
  auto read = [&](auto number, auto half, W& fw, X& fx, unsigned wring, unsigned xring) {
    constexpr int k = decltype(number)::value, h = decltype(half)::value;
    if constexpr (k < X::COUNT) fx.template read<k, h>(xring);
    else if constexpr (k < READS) fw.template read<k - X::COUNT, h>(wring);
  };
  // load number k of those that follow a step's barrier: x of a step, then weights of AHEAD
  // steps later
  auto load = [&](auto number, const auto& fromw, const auto& fromx, unsigned w0, unsigned x0) {
    constexpr int k = decltype(number)::value;
    if constexpr (k < XL) loadx(std::integral_constant<int, k>(), fromx, x0);
    else if constexpr (k < ALL) loadw(std::integral_constant<int, k - XL>(), fromw, w0);
  };
  const std::integral_constant<int, 0> first;
  const std::integral_constant<int, 1> second;
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) {
    const auto from = stepw(s);
    each<WL>([&](auto i) { loadw(i, from, s * T::WBYTES); });
  }
#pragma unroll
  for (int s = 0; s < XB - 1; ++s) {
    const auto fromw = stepw(s + AHEAD);
    const auto fromx = stepx(s);
    each<ALL>([&](auto k) { load(k, fromw, fromx, (s + AHEAD) * T::WBYTES, T::XAT + s * T::XBYTES); });
  }
  // the last buffers as if a step's barrier had been: what is over goes out in the first step
  unsigned w0 = (WB - 1) * T::WBYTES, x0 = T::XAT + (XB - 1) * T::XBYTES;
  auto fromw = stepw(WB - 1);
  auto fromx = stepx(XB - 1);
  each<NOW>([&](auto k) { load(k, fromw, fromx, w0, x0); });
  // loads that may still be on their way when the next step's have to be there
  constexpr int LATER = (AHEAD ? WL : 0) + (XB - 2) * ALL;
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(LATER + NOW) : "memory");
  each<READS>([&](auto k) { read(k, first, wa, xa, 0, 0); });
  unsigned wu = 0, xu = 0;  // this step's buffers
  // a row of products by fragments (fw, fx), reads into (gw, gx) between them
  auto row = [&](auto number, W& fw, X& fx, W& gw, X& gx, auto half, int more) {
    constexpr int i = decltype(number)::value;
    each<C>([&](auto column) {
      constexpr int j = decltype(column)::value;
      if constexpr (i == R - 1 && j == C - 1 && decltype(half)::value == 0) mul_last(acc[i][j], fw.f[i], fx.f[j], more);
      else mul(acc[i][j], fw.f[i], fx.f[j]);
      if constexpr (j == C / 2 - 1 || j == C - 1)
        each<PER>([&](auto n) { read(std::integral_constant<int, (i * 2 + (j == C - 1)) * PER + decltype(n)::value>(), half, gw, gx, wu, xu); });
    });
  };
  for (int s = 0; s < steps; ++s) {
    reads_landed();
    xa.landed();
    wa.landed();
    if (skip > 0 && s + 1 == steps) {
      xa.clear(skip, 0, threadIdx.x & 63);
      wa.clear(skip, 0, threadIdx.x & 63);
    }
    xa.whole();
    wa.whole();
    written();
    each<R>([&](auto i) {
      row(i, wa, xa, wb, xb, second, 1);
      each<LPER>([&](auto n) { load(std::integral_constant<int, NOW + decltype(i)::value * LPER + decltype(n)::value>(), fromw, fromx, w0, x0); });
      __builtin_amdgcn_sched_barrier(0);
    });
    reads_landed();
    xb.landed();
    wb.landed();
    if (skip > 0 && s + 1 == steps) {
      xb.clear(skip, 1, threadIdx.x & 63);
      wb.clear(skip, 1, threadIdx.x & 63);
    }
    xb.whole();
    wb.whole();
    written();
    // all waves have read this step, and the next one is there
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(LATER) : "memory");
    w0 = wu;
    x0 = T::XAT + xu;
    wu = wu == (WB - 1) * T::WBYTES ? 0 : wu + T::WBYTES;
    xu = xu == (XB - 1) * T::XBYTES ? 0 : xu + T::XBYTES;
    fromw = stepw(s + WB);
    fromx = stepx(s + XB);
    each<R>([&](auto i) {
      row(i, wb, xb, wa, xa, first, steps - s - 1);  // behind the last step of what nobody needs
      each<LPER>([&](auto n) {
        constexpr int k = decltype(i)::value * LPER + decltype(n)::value;
        if constexpr (k < NOW) load(std::integral_constant<int, k>(), fromw, fromx, w0, x0);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // nothing is on its way to registers or LDS
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  xa.landed();
  wa.landed();
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < C; ++j) asm volatile("" : "+a"(acc[i][j]));
  asm volatile("s_barrier" ::: "memory");
}

// A wave's results on their way out, ROWS rows of N features at a time: a lane holds four
// features of a row, whose stores would be pieces of lines; by way of LDS they are whole ones.
// 256 x 256 of bf16, all CUs at once: 8.6 us from registers, 3.4 so.
template <typename T, int N, int ROWS = 16>
struct RowsOut {
  typedef __attribute__((ext_vector_type(4))) T four_t;
  static constexpr int PER = 16 / sizeof(T), PIECES = N / PER, BYTES = ROWS * (N * sizeof(T) + 16), ROW = N * sizeof(T) + 16;  // numbers of a piece, pieces of a row
  static_assert(N % PER == 0, "");
  char* mine;
  int lane;
  DEVINL RowsOut(void* lds, int wave, int lane_) : mine((char*)lds + wave * BYTES), lane(lane_) {}
  // row `r`, features f .. f + 3
  DEVINL void put(int r, int f, four_t v) const { *(four_t*)(mine + r * ROW + f * sizeof(T)) = v; }
  // to(row, feature, piece) for all of the rows. LDS operations of a wave are in order; that lanes
  // read what others wrote, and write what others have read, is said to the compiler by the fences
  template <typename To>
  DEVINL void out(To to) const {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q0 = 0; q0 < ROWS * PIECES; q0 += 64) {
      const int q = q0 + lane, r = q / PIECES, p = q % PIECES;
      if (ROWS * PIECES % 64 == 0 || q < ROWS * PIECES) to(r, p * PER, *(const floatx4*)(mine + r * ROW + p * 16));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_sched_barrier(0);  // (the next rows' sums stay where they are meanwhile)
  }
};

// A piece to `dst`, where `there` of its numbers have a place (some may have none), in rows of N.
// Rows of bf16 that are a multiple of 4 and not of 8 go by halves: 2048 rows by [4100, 2048] took
// 52 us number by number, 41 so; 219 by [28364, 128] 17.4, 9.5
template <typename T>
DEVINL void st_piece(T* dst, floatx4 piece, int there, int N) {
  constexpr int PER = 16 / sizeof(T);
  typedef __attribute__((ext_vector_type(2))) float floatx2;
  if (N % PER == 0 && there >= PER) *(floatx4*)dst = piece;
  else if (sizeof(T) == 2 && N % 4 == 0) {
    if (there >= 4) *(floatx2*)dst = (floatx2){piece[0], piece[1]};
    if (there >= 8) *(floatx2*)(dst + 4) = (floatx2){piece[2], piece[3]};
  } else {
    union { floatx4 v; T e[PER]; } u = {piece};
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (i < there) dst[i] = u.e[i];
  }
}
