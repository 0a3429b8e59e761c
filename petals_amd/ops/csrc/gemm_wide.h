// A tile of X [M, K] times W [K, N], or W [N, K] transposed, in bf16, by four waves with one SIMD each: the
// core of the products of hundreds of rows, for whoever says where rows and columns lie.
//
// Up to 256 x 256 values are a workgroup's, and a wave's 512 registers hold 64 x 4 of their sums: eight waves
// with a quarter as many each read fragments 1.5 times as often, and LDS reads and the loads that fill it kept
// that form at 1.1 PFLOP/s. One wave has nobody to fill its gaps, so its loads, LDS reads and products are issued in
// a fixed order: a group of FN products for each fragment of X, what is read or loaded meanwhile spread among them
// (all of it ahead of a group's products: 6% slower). K goes in steps of 64, in two halves of 32: products of one
// half, fragments of W of the next, those of X three groups ahead.
//
// What bounds it is the way from L2 to LDS, 50 KB a us for a compute unit, and the time loads have to come back:
// LDS holds three stages of X and two of W, or three where they fit. A barrier ahead of each half frees what was read in the
// one before, so that loads are spread over the whole step and have one to one and a half steps. With
// one barrier a step and all loads behind it: 4096 x 4096 x 28672 took 767 us and not 728 (1.32 PFLOP/s, the
// library's 743), 758 x 22016 x 4096 transposed 131 and not 119.
//
// W [K, N] is read by transposing loads. Weights straight to registers instead of LDS needed twice the
// loads (8 bytes a lane), and conversions that a wave without a partner can't hide: 7% slower, transposed 30%.
//
// The matrix instructions are in asm: their sums stay in one register each there, where the compiler moved
// a third of them about in every step. It does not see their hazards, so: operands come from LDS loads only, whose
// waits it does see; sums are set before a barrier; and none is read within 32 cycles after the last one. Nor may it copy or
// spill a sum within a loop. ops/sums_check.py looks at what was built for all of this, and the build fails if it isn't so.
#pragma once

#include "gemm.h"
#include <type_traits>
#include <utility>

#define WIDE_THREADS 256

template <int... I, class F>
__device__ __forceinline__ void wide_each(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void wide_each(F&& f) {
  wide_each(std::make_integer_sequence<int, N>{}, f);
}

// WR x 4 / WR waves of 16 FM rows and 16 FN columns
template <bool WT, int WR, int FM, int FN>
struct WideTile {
  static constexpr int WC = 4 / WR, BM = WR * FM * 16, BN = WC * FN * 16, BK = 64;
  static constexpr int XB = BM * BK * 2, WB = BN * BK * 2;                           // bytes of a stage
  static constexpr int SX = 3, SW = SX * XB + 3 * WB <= 160 * 1024 ? 3 : 2;          // stages
  static constexpr int LDS = SX * XB + SW * WB;
  static_assert(FM * FN <= 64 && FN % 2 == 0 && LDS <= 160 * 1024);
};

// sums past the 56th are in ordinary registers: with all 64 x 4 in the accumulation registers none is left to
// move them through
template <bool ACCUMULATION>
__device__ __forceinline__ void wide_mfma(f32x4& sum, bf16x8 a, bf16x8 b) {
  if constexpr (ACCUMULATION)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(sum) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(sum) : "v"(a), "v"(b));
}
// keeps reads of the accumulation registers where they are used, which else take all other registers at once
template <bool ACCUMULATION>
__device__ __forceinline__ void wide_pin(f32x4& sum) {
  if constexpr (ACCUMULATION) asm volatile("" : "+a"(sum));
}

__device__ __forceinline__ gemm_rsrc wide_resource(const void* p, unsigned bytes) {
  const size_t at = (size_t)p;
  return gemm_rsrc{__builtin_amdgcn_readfirstlane((int)at), __builtin_amdgcn_readfirstlane((int)(at >> 32) & 0xFFFF),
                   (int)bytes, 0x00020000};
}

// byte offset of 16-byte group c in a row of 128 bytes, and what is added to the group in a row of W [K, N]
__device__ __forceinline__ int wide_group(int row, int c) { return row * 128 + ((c ^ (row & 7)) << 4); }
template <int BN>
__device__ __forceinline__ int wide_swizzle(int row) {
  static_assert(BN % 64 == 0 && BN >= 128);
  constexpr int GROUPS = BN % 128 ? 8 : 16;  // that are permuted among themselves
  return ((row & 3) | ((row >> 1) & 4)) << 1 & (GROUPS - 1);
}

// acc[i][j]: sums of `steps` steps from `first` on; 4 neighbouring columns, hi * 4 of fragment i, of row lane % 16 of
// fragment j. x_row(row of the tile): byte offset of that row in x. w_at(c): which column of W the tile's c is;
// for W [K, N] c is a multiple of 8 and so are 8 columns there. row_bytes: of a row of W.
template <bool WT, int WR, int FM, int FN, class XRow, class WAt>
__device__ __forceinline__ void wide_product(
    unsigned char* lds, f32x4 (&acc)[FN][FM], gemm_rsrc xr, gemm_rsrc wr, XRow x_row, WAt w_at,
    unsigned row_bytes, int first, int steps) {
  using Tile = WideTile<WT, WR, FM, FN>;
  constexpr int WC = Tile::WC, BK = Tile::BK, BN = Tile::BN, XB = Tile::XB, WB = Tile::WB, SX = Tile::SX, SW = Tile::SW;
  constexpr int G = 2 * FM;                                                      // groups of a step
  constexpr int WIN = G <= 8 ? G : G % 8 == 0 ? 8 : G % 10 == 0 ? 10 : G % 7 == 0 ? 7 : 6;  // fragments of X
  static_assert(G % WIN == 0);
  // groups that they are read ahead: some 24 products
  constexpr int AHEAD = (24 + FN - 1) / FN, D = AHEAD < FM && AHEAD < WIN - 1 ? AHEAD : FM < WIN - 1 ? FM : WIN - 2 > 0 ? WIN - 2 : 1;
  static_assert(D < WIN && D <= FM);
  constexpr int XL = XB / 4096, WL = WB / 4096;                                   // loads of 1 KB of a step, per wave
  constexpr int XA = WT ? XL : (XL + 1) / 2, WA = WT ? 0 : WL / 2;                    // of its first half

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid & (WAVE - 1);
  const int col = lane & 15, hi = lane >> 4;
  const int wm = wave / WC * FM * 16, wn = wave % WC * FN * 16;
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds, wbase = base + SX * XB;

  // a load's place in its stage; the first half of a wave's loads of W [K, N] are of the first 32 rows
  auto x_load = [&](int i) { return wave * XL + i; };
  auto w_load = [&](int i) { return WT ? wave * WL + i : i / (WL / 2) * (WL * 2) + wave * (WL / 2) + i % (WL / 2); };
  unsigned x_lane[XL], w_lane[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int p = x_load(i) * 64 + lane, row = p / 8;
    x_lane[i] = x_row(row) + (p % 8 ^ (row & 7)) * 16;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int p = w_load(i) * 64 + lane, row = p / (WT ? 8 : BN / 8);
    w_lane[i] = WT ? w_at(row) * row_bytes + (p % 8 ^ (row & 7)) * 16
                   : row * row_bytes + w_at((p % (BN / 8) ^ wide_swizzle<BN>(row)) * 8) * 2;
  }
  const unsigned w_step = WT ? BK * 2 : BK * row_bytes;
  auto load = [&](unsigned to, unsigned from, gemm_rsrc r, unsigned at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(to), "v"(from), "s"(r), "s"(at)
                 : "memory", "m0");
  };
  // stages are byte offsets: those that are read, those that are filled and the steps that these get. Past
  // the end the last step is loaded again, to stages that nobody reads any more.
  auto next = [](unsigned at, unsigned size, int n) { return at + size == size * n ? 0u : at + size; };
  unsigned x_from = 0, w_from = 0, x_to = 0, w_to = 0;
  int x_new = 0, w_new = 0;
  auto load_x = [&](int i) { load(base + x_to + x_load(i) * 1024, x_lane[i], xr, (unsigned)(first + min(x_new, steps - 1)) * (BK * 2)); };
  auto load_w = [&](int i) { load(wbase + w_to + w_load(i) * 1024, w_lane[i], wr, (unsigned)(first + min(w_new, steps - 1)) * w_step); };
  auto x_done = [&] { x_to = next(x_to, XB, SX), ++x_new; };
  auto w_done = [&] { w_to = next(w_to, WB, SW), ++w_new; };

  using lds_v4s = __attribute__((address_space(3))) v4s;
  using lds_frag = const __attribute__((address_space(3))) bf16x8;
  unsigned xa[2], wa[WT ? 2 : FN];  // addresses of this lane's fragments
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    xa[h] = base + wide_group(wm + col, h * 4 + hi);
    if (WT) wa[h] = wbase + wide_group(wn + col, h * 4 + hi);
  }
  if (!WT)
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int row = hi * 8 + col / 4, c = (wn + i * 16) / 8 + ((col >> 1) & 1);
      wa[i] = wbase + row * (BN * 2) + ((c ^ wide_swizzle<BN>(row)) << 4) + (col & 1) * 8;
    }
  bf16x8 wf[2][FN], xf[WIN];
  auto read_x = [&](unsigned from, int g) { xf[g % WIN] = *(lds_frag*)(size_t)(xa[g / FM] + from + g % FM * (16 * 128)); };
  auto read_w = [&](unsigned from, int h, int i) {
    if (WT) {
      wf[h][i] = *(lds_frag*)(size_t)(wa[h] + from + i * (16 * 128));
    } else {
      // rows hi * 8 + col / 4 and 4 below, which are permuted alike; 4 columns a lane
      const unsigned p = wa[i] + from + h * 32 * BN * 2;
      const v4s a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(size_t)p);
      const v4s b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(size_t)(p + 4 * BN * 2));
      wf[h][i] = bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    }
  };

#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SW; ++s) {
    if (s < 2) {
#pragma unroll
      for (int i = 0; i < XL; ++i) load_x(i);
      x_done();
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) load_w(i);
    w_done();
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XL + (SW - 1) * WL) : "memory");  // step 0 is there
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < FN; ++i) read_w(0, 0, i);
#pragma unroll
  for (int g = 0; g < D; ++g) read_x(0, g);
  __builtin_amdgcn_sched_barrier(0);

  // Loads of step t: X of t + 2 in its first half (W [N, K]) or in both, W of t + SW in both or in the second.
  int t = 0;
  do {
    const unsigned x_next = next(x_from, XB, SX), w_next = next(w_from, WB, SW);
    wide_each<G>([&](auto g_) {
      constexpr int g = decltype(g_)::value, h = g / FM, j = g % FM;
      if constexpr (j == 0) {
        // What this half reads is there: W of the next half, and in the second X of the next step. All waves have read
        // what its loads overwrite, up to their last fragment of X: X of the step before; of W the whole step
        // in the second half, or the rows of this half. Loads come back in order; `out` were issued later.
        constexpr int out = WT ? (h ? XL + (SW - 2) * WL : 63) : h ? XA + WL : XL + WL;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(1)" ::"n"(out) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      // in the order of issue: fragments of W, one of X, loads
      constexpr int w0 = j * FN / FM, ws = (j + 1) * FN / FM - w0;
      constexpr int xs = h ? XL - XA : XA, all = xs + (h ? WL - WA : WA);
      constexpr int l0 = j * all / FM, l1 = (j + 1) * all / FM, ops = ws + 1 + l1 - l0;
      wide_each<FN>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        wide_each<ops>([&](auto o_) {
          constexpr int o = decltype(o_)::value;
          if constexpr (o * FN / ops == i) {
            if constexpr (o < ws) {
              read_w(h ? w_next : w_from, h ^ 1, w0 + o);
            } else if constexpr (o == ws) {
              if constexpr (g + D < G) read_x(x_from, g + D);
              else read_x(x_next, g + D - G);
            } else {
              constexpr int l = l0 + o - 1 - ws;
              if constexpr (l < xs) load_x(h ? XA + l : l);
              else load_w((h ? WA : 0) + l - xs);
            }
          }
        });
        wide_mfma<(j * FN + i < 56)>(acc[i][j], wf[h][i], xf[g % WIN]);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    x_done();
    w_done();
    x_from = x_next;
    w_from = w_next;
  } while (++t < steps);
  // no load is on its way when LDS gets another owner
  asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Two fragments of neighbouring columns -> 8 columns of one row a lane: of the first one for even hi and of the second
// for odd, from (hi / 2) * 8 on. All lanes take part.
__device__ __forceinline__ void wide_join(f32x4 a, f32x4 b, float (&v)[8]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const auto u = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[r]), __float_as_uint(b[r]), false, false);
    v[r] = __uint_as_float(u[0]);
    v[r + 4] = __uint_as_float(u[1]);
  }
}

// a lane's row and column of a wave's tile, for the first of its groups of 8 columns
template <bool WT, int WR, int FM, int FN>
__device__ __forceinline__ int wide_row() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) / WideTile<WT, WR, FM, FN>::WC * FM * 16 + (threadIdx.x & 15);
}
template <bool WT, int WR, int FM, int FN>
__device__ __forceinline__ int wide_column() {
  using Tile = WideTile<WT, WR, FM, FN>;
  const int hi = (threadIdx.x & (WAVE - 1)) >> 4;
  return __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) % Tile::WC * FN * 16 + (hi & 1) * 16 + (hi >> 1) * 8;
}

// store(j, i, 8 values) for all of a lane's groups: of row wide_row() + 16 j and columns from wide_column() + 32 i on.
// `pairs`: store(j, i, gates, ups), the first half of a wave's columns being gates. ahead(j) is called a row
// earlier: what it loads is on its way while that one is stored.
template <int FM, int FN, class Ahead, class Store>
__device__ __forceinline__ void wide_store(bool pairs, f32x4 (&acc)[FN][FM], Ahead ahead, Store store) {
  ahead(std::integral_constant<int, 0>{});
  wide_each<FM>([&](auto j) {
    if constexpr (j + 1 < FM) ahead(std::integral_constant<int, j + 1>{});
    wide_each<FN>([&](auto i) { wide_pin<(j * FN + i < 56)>(acc[i][j]); });
    // halves of an odd number of pairs are nobody's: their callers have none
    if (pairs && FN % 4 == 0) {
      wide_each<FN / 4>([&](auto i) {
        float g[8], u[8];
        wide_join(acc[2 * i][j], acc[2 * i + 1][j], g);
        wide_join(acc[2 * i + FN / 2][j], acc[2 * i + 1 + FN / 2][j], u);
        store(j, i, g, u);
      });
    } else {
      wide_each<FN / 2>([&](auto i) {
        float v[8];
        wide_join(acc[2 * i][j], acc[2 * i + 1][j], v);
        store(j, i, v, v);
      });
    }
  });
}
