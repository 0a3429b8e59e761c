// What the products of a prompt's rows share, whatever holds the weights: tiles and parts of a product, its
// plan, and what follows it.
#pragma once

#include "common.h"
#include "gemv_reduce.h"
#include "paged.h"

#define GEMM_THREADS 512
#define GEMM_CUS 256

enum GemmEpilogue : int {
  GEMM_PLAIN = 0,     // y
  GEMM_RESIDUAL = 1,  // residual + y + bias
  GEMM_GELU = 2,      // gelu(y + bias)
  GEMM_SWIGLU = 3,    // silu(y[:N/2]) * y[N/2:]
};

struct GemmShape {
  int m, n, k;
  int row_tiles;  // of a run of columns
  int band;       // of these that follow each other before the next run of columns
  int whole;      // tiles summed over all of K
  int rest;       // tiles split along K
  int splits, per;  // parts of these, and steps of each
};

struct GemmOut {
  unsigned short* y;               // [M, N], or [M, N/2] for GEMM_SWIGLU
  const unsigned short* residual;  // [M, N] or null
  const unsigned short* bias;      // [N] or null
  float* parts;                    // [splits, rest, BM, BN]
  int epilogue;
};

using u32x4 = __attribute__((ext_vector_type(4))) unsigned;
using gemm_rsrc = __attribute__((ext_vector_type(4))) int;

// where a tile's column comes from: with GEMM_SWIGLU, half of a wave's columns are gates, and
// the other half the same columns of up
template <int FN>
__device__ __forceinline__ int gemm_source_column(int tile, int c, int bn, int n, bool pairs) {
  if (!pairs) return tile * bn + c;
  constexpr int HALF = FN * 8;
  const int in = c % (2 * HALF);
  return tile * (bn / 2) + c / (2 * HALF) * HALF + in % HALF + (in >= HALF ? n / 2 : 0);
}

// four neighbouring values of a row, at column c of y's
__device__ __forceinline__ void gemm_store(const GemmShape& s, const GemmOut& o, int m, int c, f32x4 v) {
  if (m >= s.m || c >= s.n) return;
  if (o.bias) {
    const v4s b = *reinterpret_cast<const v4s*>(o.bias + c);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += bf16_to_f32((unsigned short)b[i]);
  }
  const size_t at = (size_t)m * s.n + c;
  if (o.residual) {
    const v4s r = *reinterpret_cast<const v4s*>(o.residual + at);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += bf16_to_f32((unsigned short)r[i]);
  }
  v4s y;
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = (short)f32_to_bf16(o.epilogue == GEMM_GELU ? gelu_tanh_f32(v[i]) : v[i]);
  *reinterpret_cast<v4s*>(o.y + at) = y;
}

__device__ __forceinline__ void gemm_store_pair(const GemmShape& s, const GemmOut& o, int m, int c, f32x4 g, f32x4 u) {
  if (m >= s.m || c >= s.n / 2) return;
  v4s y;
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = (short)f32_to_bf16(g[i] / (1.f + __expf(-g[i])) * u[i]);
  *reinterpret_cast<v4s*>(o.y + (size_t)m * (s.n / 2) + c) = y;
}

// 8 values of a bias or a residual, which are aligned to 8 bytes
struct Gemm8 {
  v4s v[2];
};
__device__ __forceinline__ Gemm8 gemm_load8(const unsigned short* p) {
  return {reinterpret_cast<const v4s*>(p)[0], reinterpret_cast<const v4s*>(p)[1]};
}

// the same for 8 values, in 16-byte groups, with a bias and a residual that are there already
__device__ __forceinline__ void gemm_store(
    const GemmShape& s, const GemmOut& o, int m, int c, float (&v)[8], const Gemm8& bias, const Gemm8& residual) {
  if (m >= s.m || c >= s.n) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (o.bias) v[i] += bf16_to_f32((unsigned short)bias.v[i / 4][i % 4]);
    if (o.residual) v[i] += bf16_to_f32((unsigned short)residual.v[i / 4][i % 4]);
    if (o.epilogue == GEMM_GELU) v[i] = gelu_tanh_f32(v[i]);
  }
  store8(o.y + (size_t)m * s.n + c, v);
}

__device__ __forceinline__ void gemm_store_pair(const GemmShape& s, const GemmOut& o, int m, int c, float (&g)[8], float (&u)[8]) {
  if (m >= s.m || c >= s.n / 2) return;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = g[i] / (1.f + __expf(-g[i])) * u[i];
  store8(o.y + (size_t)m * (s.n / 2) + c, v);
}

// where a tile lies. Bands of rows bound what a chiplet's 32 workgroups read of X for each of their runs of columns:
// 4096 x 4096 x 28672 in tiles of 256 rows took 3% longer with 16 of them below each other than with 8.
struct GemmPlace {
  int row, column;  // in tiles
};
template <int BN>
__device__ __forceinline__ GemmPlace gemm_place(const GemmShape& s, int tile) {
  if (s.band == s.row_tiles) return {tile % s.row_tiles, tile / s.row_tiles};
  const int all = (s.n + BN - 1) / BN * s.band, above = tile / all * s.band, in = tile % all, rows = min(s.band, s.row_tiles - above);
  return {above + in % rows, in / rows};
}

// a workgroup's tile, and its steps of `all`: each chiplet has a run of its own. part: -1 for a sum over
// all of K. False: none, for the whole workgroup.
struct GemmSpot {
  int tile, first, steps, part;
};
__device__ __forceinline__ bool gemm_spot(const GemmShape& s, int all, GemmSpot* spot) {
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  if (local < s.whole / 8) {  // `whole` is a multiple of 8
    *spot = {xcd * (s.whole / 8) + local, 0, all, -1};
    return true;
  }
  const int units = s.rest * s.splits, share = (units + 7) / 8, unit = xcd * share + local - s.whole / 8;
  if (local - s.whole / 8 >= share || unit >= units) return false;
  const int first = unit / s.rest * s.per;
  *spot = {s.whole + unit % s.rest, first, min(s.per, all - first), s.splits > 1 ? unit / s.rest : -1};
  return true;
}

// four values of a tile per thread
template <int BM, int BN, int FN>
__global__ __launch_bounds__(256) void gemm_parts_kernel(GemmShape s, GemmOut o) {
  const bool pairs = o.epilogue == GEMM_SWIGLU;
  const int at = blockIdx.x * 256 + threadIdx.x, columns = pairs ? BN / 2 : BN;
  const int tile = at / (BM * columns / 4), in = at % (BM * columns / 4) * 4;
  if (tile >= s.rest) return;
  const int row = in / columns;
  int c = in % columns;
  if (pairs) c = c / (FN * 8) * (FN * 16) + c % (FN * 8);
  const GemmPlace place = gemm_place<BN>(s, s.whole + tile);
  const int m = place.row * BM + row, column_tile = place.column;
  if (m >= s.m) return;
  const float* p = o.parts + (size_t)tile * (BM * BN) + row * BN + c;
  const size_t stride = (size_t)s.rest * (BM * BN);
  f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f}, up = sum;
  for (int i = 0; i < s.splits; ++i) {
    sum += *reinterpret_cast<const f32x4*>(p + i * stride);
    if (pairs) up += *reinterpret_cast<const f32x4*>(p + i * stride + FN * 8);
  }
  const int n = gemm_source_column<FN>(column_tile, c, BN, s.n, pairs);
  if (pairs) gemm_store_pair(s, o, m, n, sum, up);
  else gemm_store(s, o, m, n, sum);
}

struct GemmTile {
  int bm, bn;
  float step;  // us of a step, a tile on every compute unit
  // us of a tile beside its steps; share of a step's time that is left with few tiles
  float fixed = 0.f, alone = 1.f;
};

// tiles of a product in steps of bk, parts of at least `least` of them
static GemmShape gemm_plan(long m, long n, long k, int bk, long least, const GemmTile& t, float* us) {
  const long row_tiles = (m + t.bm - 1) / t.bm, tiles = row_tiles * ((n + t.bn - 1) / t.bn), steps = k / bk;
  long whole = tiles / GEMM_CUS * GEMM_CUS, rest = tiles - whole, splits = 1;
  if (rest) splits = std::max(1L, std::min(GEMM_CUS / rest, steps / least));
  long per = (steps + splits - 1) / splits;
  splits = (steps + per - 1) / per;
  *us = tiles / GEMM_CUS * (t.step * steps + t.fixed);
  if (rest) *us += t.step * per * (t.alone + (1.f - t.alone) * rest * splits / GEMM_CUS) + t.fixed;
  if (splits > 1) *us += 5.f + rest * splits * t.bm * t.bn * 4 * 2 / 8e6f;
  const long bands = (row_tiles * t.bm + 2047) / 2048, band = (row_tiles + bands - 1) / bands;
  return GemmShape{(int)m, (int)n, (int)k, (int)row_tiles, (int)band, (int)whole, (int)rest, (int)splits, (int)per};
}
