// Device-routed MoE expert GEMVs for CDNA4 (gfx950).
//
// Decode-time grouped GEMM: virtual row r = (token b = r/K, slot j = r%K)
// reads its expert id from a DEVICE tensor (written by the on-GPU router:
// softmax + top-k, no host sync) and streams that expert's stacked weights.
// Everything is hipGraph-capturable — the expert choice is data in device
// buffers, not launch parameters — which is what lets Mixtral spans use the
// whole-span decode graph (the reference runs Mixtral experts densely inside
// HF code with host-side routing: reference models/mixtral/block.py:73-81).
//
// Weight layouts match gemv.hip / nf4_tiles.hip, stacked on a leading expert axis:
//   bf16: wt_all   [E, in, out]
//   nf4:  tiles    [E, out/64, in/128, 4, 64, 16], scales [E, out/64, in]; its GEMV is
//         nf4_tiles.hip's
// The per-row inner loop is the same x-broadcast split-K structure as the
// dense kernels (each selected expert's weights are read exactly once per
// token); experts whose rows are aligned to 16 bytes take gemv_mfma.h's.

#include "common.h"
#include "gemm_wide.h"
#include "gemv_mfma.h"
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

#ifndef GEMV_OUT_PER_WAVE
#define GEMV_OUT_PER_WAVE 512
#endif

using bf16x8_moe = __attribute__((ext_vector_type(8))) short;
using f32x4_moe = __attribute__((ext_vector_type(4))) float;

static __device__ __constant__ float MOE_NF4_LUT[16] = {
    -1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f,
    -0.28444138169288635f, -0.18477343022823334f, -0.09105003625154495f, 0.0f,
    0.07958029955625534f, 0.16093020141124725f, 0.24611230194568634f,
    0.33791524171829224f, 0.4407098293304443f, 0.5626170039176941f,
    0.7229568362236023f, 1.0f};

// ------------------------------------------------------------ bf16 indexed

__global__ __launch_bounds__(WAVE) void gemv_bf16_moe_kernel(
    const unsigned short* __restrict__ wt_all,  // [E, in, out]
    const float* __restrict__ x,                // [B, in]
    const int* __restrict__ sel,                // [R] expert per virtual row
    float* __restrict__ partials,               // [n_splits, R, out]
    int in_dim,
    int out_dim,
    int i_per_split,
    int rows,
    int k_per_tok) {
  const int row = blockIdx.z;
  const int lane = threadIdx.x & (WAVE - 1);
  const int out0 = blockIdx.x * GEMV_OUT_PER_WAVE + lane * 8;
  if (out0 >= out_dim) return;
  const int split = blockIdx.y;
  const int i_begin = split * i_per_split;
  const int i_end = min(i_begin + i_per_split, in_dim);

  const int e = sel[row];
  const unsigned short* wt = wt_all + (size_t)e * in_dim * out_dim;
  const float* xr = x + (size_t)(row / k_per_tok) * in_dim;

  float acc[8];
#pragma unroll
  for (int v = 0; v < 8; ++v) acc[v] = 0.f;

  const bool full = (out0 + 8) <= out_dim;
  if (full) {
    constexpr int UNROLL = 16;
    const unsigned short* wp = wt + (size_t)i_begin * out_dim + out0;
    int i = i_begin;
    for (; i + UNROLL <= i_end; i += UNROLL) {
      short8 w8[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
        w8[u] = *reinterpret_cast<const short8*>(wp + (size_t)u * out_dim);
      float xs[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) xs[u] = xr[i + u];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
#pragma unroll
        for (int v = 0; v < 8; ++v)
          acc[v] = fmaf(bf16_to_f32((unsigned short)w8[u][v]), xs[u], acc[v]);
      }
      wp += (size_t)UNROLL * out_dim;
    }
    for (; i < i_end; ++i) {
      const short8 w8 = *reinterpret_cast<const short8*>(wt + (size_t)i * out_dim + out0);
      const float xv = xr[i];
#pragma unroll
      for (int v = 0; v < 8; ++v) acc[v] = fmaf(bf16_to_f32((unsigned short)w8[v]), xv, acc[v]);
    }
  } else {
    for (int i = i_begin; i < i_end; ++i) {
      const float xv = xr[i];
#pragma unroll
      for (int v = 0; v < 8; ++v)
        if (out0 + v < out_dim)
          acc[v] = fmaf(bf16_to_f32(wt[(size_t)i * out_dim + out0 + v]), xv, acc[v]);
    }
  }

  float* dst = partials + ((size_t)split * rows + row) * out_dim + out0;
  if (full) {
    float4v* d4 = reinterpret_cast<float4v*>(dst);
    d4[0] = float4v{acc[0], acc[1], acc[2], acc[3]};
    d4[1] = float4v{acc[4], acc[5], acc[6], acc[7]};
  } else {
#pragma unroll
    for (int v = 0; v < 8; ++v)
      if (out0 + v < out_dim) dst[v] = acc[v];
  }
}

// ------------------------------------------------------------- routing
//
// A token's router, softmax, choice and renormalization in one launch, its experts' sum
// and the residual in another: as torch operations they were 12 and 5 launches of 4 to 20
// us each (the selection alone 19), half of a decoding step of two Mixtral 8x7B blocks.

#define ROUTE_EXPERTS 256  // at most
#define ROUTE_TOP 16

// One token per workgroup: 4 waves take every fourth expert.
template <typename T>
__global__ __launch_bounds__(256) void moe_route_kernel(
    const T* __restrict__ x,                // [tokens, dim]
    const unsigned short* __restrict__ w,   // [experts, dim] bf16
    float* __restrict__ weights, int* __restrict__ sel, int dim, int experts, int top) {
  __shared__ float logits[ROUTE_EXPERTS];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid & (WAVE - 1);
  const T* row = x + (size_t)blockIdx.x * dim;
  for (int e = wave; e < experts; e += 4) {
    float sum = 0.f;
    for (int c = lane * 8; c < dim; c += WAVE * 8) {
      float a[8], b[8];
      load8(row + c, a);
      load8(w + (size_t)e * dim + c, b);
#pragma unroll
      for (int i = 0; i < 8; ++i) sum = fmaf(a[i], b[i], sum);
    }
    sum = wave_reduce_sum(sum);
    if (lane == 0) logits[e] = sum;
  }
  __syncthreads();
  if (wave != 0) return;
  // Of this lane's experts; chosen ones drop out. A softmax of infinities or NaNs has NaNs for
  // all, but for logits below every number among others: those count as just above the sentinel.
  float v[ROUTE_EXPERTS / WAVE];
  bool odd = false, some = false;
#pragma unroll
  for (int i = 0; i < ROUTE_EXPERTS / WAVE; ++i) {
    v[i] = NEG_SENTINEL;
    if (lane + i * WAVE >= experts) continue;
    const unsigned bits = __float_as_uint(logits[lane + i * WAVE]);
    const bool finite = (bits & 0x7FFFFFFFu) < 0x7F800000u;
    odd |= !finite && bits != 0xFF800000u;
    some |= finite;
    v[i] = finite ? fmaxf(__uint_as_float(bits), NEG_THRESHOLD) : NEG_THRESHOLD;
  }
  odd = __any(odd) || !__any(some);
  float first = 0.f, total = 0.f, mine = 0.f;
  int chosen = 0;
  for (int j = 0; j < top; ++j) {
    float best = v[0];
    int at = lane;
#pragma unroll
    for (int i = 1; i < ROUTE_EXPERTS / WAVE; ++i)
      if (v[i] > best) best = v[i], at = lane + i * WAVE;
    if (at >= experts) at = 0;  // nothing left here
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float other = __shfl_xor(best, off, WAVE);
      const int where = __shfl_xor(at, off, WAVE);
      if (other > best || (other == best && where < at)) best = other, at = where;
    }
#pragma unroll
    for (int i = 0; i < ROUTE_EXPERTS / WAVE; ++i)
      if (at == lane + i * WAVE) v[i] = NEG_SENTINEL;
    if (j == 0) first = best;
    const float p = __expf(best - first);  // of the softmax over all, up to the factor that cancels
    total += p;
    if (lane == j) mine = p, chosen = at;
  }
  if (lane < top) {
    weights[(size_t)blockIdx.x * top + lane] = odd ? __uint_as_float(0x7FC00000u) : mine / total;
    sel[(size_t)blockIdx.x * top + lane] = chosen;
  }
}

// y[b] = residual[b] + sum_j weights[b, j] * (sum over splits of partials[:, b * top + j]);
// 64 outputs by 16 groups of (split, slot) per workgroup
__global__ __launch_bounds__(1024) void moe_reduce_kernel(
    const float* __restrict__ partials,  // [splits, tokens * top, out]
    const float* __restrict__ weights, const unsigned short* __restrict__ residual, unsigned short* __restrict__ y,
    int splits, int tokens, int top, int out_dim) {
  __shared__ float part[16][64];
  const int c = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int o = blockIdx.x * 64 + c, b = blockIdx.y;
  float sum = 0.f;
  if (o < out_dim)
    for (int i = g; i < splits * top; i += 16) {
      const int s = i / top, j = i - s * top;
      sum = fmaf(weights[b * top + j], partials[((size_t)s * tokens * top + b * top + j) * out_dim + o], sum);
    }
  part[g][c] = sum;
  __syncthreads();
  if (g != 0 || o >= out_dim) return;
  sum = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) sum += part[i][c];
  y[(size_t)b * out_dim + o] = f32_to_bf16(bf16_to_f32(residual[(size_t)b * out_dim + o]) + sum);
}

// the same for rows [tokens * top, out] in bf16, 8 values per thread
__global__ __launch_bounds__(256) void moe_combine_kernel(
    const unsigned short* __restrict__ rows, const float* __restrict__ weights, const unsigned short* __restrict__ residual,
    unsigned short* __restrict__ y, int top, int out_dim, long groups) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  if (g >= groups) return;
  const long t = g * 8 / out_dim, c = g * 8 - t * out_dim;
  float sum[8], v[8];
  load8(residual + g * 8, sum);
  for (int j = 0; j < top; ++j) {
    load8(rows + (t * top + j) * out_dim + c, v);
    const float w = weights[t * top + j];
#pragma unroll
    for (int i = 0; i < 8; ++i) sum[i] = fmaf(w, v[i], sum[i]);
  }
  store8(y + g * 8, sum);
}

// One workgroup. counts -> padded offsets -> scatter; every sorted slot and
// every tile is written. The order of an expert's pairs is not fixed, which no
// result depends on (each pair is a row of its own).
__global__ __launch_bounds__(1024) void moe_group_kernel(
    const int* __restrict__ sel, int pairs, int experts, int mt, int slots,
    int* __restrict__ sorted_pairs, int* __restrict__ tile_expert) {
  extern __shared__ int cnt[];  // [experts] counts, then next free slot
  int* end = cnt + experts;     // [experts] end of the padded segment
  const int tid = threadIdx.x;
  for (int e = tid; e < experts; e += blockDim.x) cnt[e] = 0;
  for (int i = tid; i < slots; i += blockDim.x) sorted_pairs[i] = -1;
  for (int i = tid; i < slots / mt; i += blockDim.x) tile_expert[i] = -1;
  __syncthreads();
  for (int i = tid; i < pairs; i += blockDim.x) {
    const int e = sel[i];
    if (e >= 0 && e < experts) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (tid == 0) {
    int at = 0;
    for (int e = 0; e < experts; ++e) {
      const int padded = (cnt[e] + mt - 1) / mt * mt;
      cnt[e] = at;
      at += padded;
      end[e] = at;
    }
  }
  __syncthreads();
  for (int e = tid; e < experts; e += blockDim.x)
    for (int i = cnt[e]; i < end[e]; i += mt) tile_expert[i / mt] = e;
  __syncthreads();
  for (int i = tid; i < pairs; i += blockDim.x) {
    const int e = sel[i];
    if (e >= 0 && e < experts) sorted_pairs[atomicAdd(&cnt[e], 1)] = i;
  }
}

// ------------------------------------------------- grouped GEMM (prefill)
//
// Grouped GEMM over expert-sorted (token, slot) pairs: the caller sorts the R = T*k
// pairs by expert with each expert's segment padded to a multiple of MT rows, so every
// MT-row tile belongs to ONE expert (tile_expert[tile], -1 = pure padding).
//
// NF4 weights, and bf16 beyond offsets of 32 bits or where a call asks for it (the others: moe_wide_kernel below).
// Up to four tiles of one expert (128 rows) and 256 columns are a workgroup's: an
// expert's weights are read once per 128 of its rows, and the rows once per 256 columns.
// With a tile of 32 rows and 128 columns each, weights crossed the caches four times as
// often and every product waited for a transposing store of its weights. Both products of
// a layer of 8 experts, width 4096 and inner size 14336: with 290 rows an expert from 6.06
// to 1.20 ms (135 to 680 TFLOP/s), with 71 from 2.09 to 0.57 ms (weights at 5.0 TB/s).
//
// 8 waves of 64 x 64, two on a SIMD; K in steps of 64 through two LDS buffers. The two
// waves of a SIMD take turns, half a step apart: while one moves (fragments out of LDS, the
// next step's tile into it), the other keeps the matrix cores busy and asks for the tile
// after next but one. All in step, with both halves of a step's fragments read ahead:
// 1.33 and 0.61 ms; fragments read as they were needed and loads one step ahead: 1.73 and
// 0.80 ms, 58% of all wave time spent waiting (with NF4 weights 2.31 to 2.02 ms with 290
// rows, 0.96 to 0.86 ms with 71). Loads have no conditions, rows and columns
// beyond the end repeat the last: with a condition on one of them the compiler can't tell
// how many are in flight and waits for all. Tiles of 256 rows, of 128 columns with two
// workgroups on a CU, and steps of 32 were all slower.
//
// The product is W^T X^T, so that a lane ends with 4 neighbouring columns of one row.
// Weights in bf16 lie in LDS as in memory and are read by transposing loads. NF4 weights
// are dequantized on the way, so that their packed form is what is read: a thread has 16
// codes of one column, and its LDS rows are columns. The 16-byte groups of an LDS row, of
// 128 or (W in bf16) 512 bytes, are permuted by the row, so that the 16 rows that a load
// touches lie in different banks.
//
// Workgroups are dealt to the 8 chiplets in turn; a chiplet takes every eighth run of
// columns. Up to MOE_SHARE row groups of an expert follow each other with the same run:
// they find its weights in the chiplet's L2, and the next run finds their rows there
// (2 to 5% over all groups of all experts with one run).

#define MOE_MT 32    // rows of a tile of one expert
#define MOE_BM 128   // rows of a workgroup
#define MOE_BN 256   // columns of a workgroup
#define MOE_BK 64    // k step
#define MOE_SHARE 8  // row groups that share a run of columns

// where 16-byte group c of a row lies
__device__ __forceinline__ int moe_x_at(int row, int c) { return row * (MOE_BK * 2) + ((c ^ ((row >> 1) & 7)) << 4); }
__device__ __forceinline__ int moe_w_at(int row, int c) {
  return row * (MOE_BN * 2) + ((c ^ (((row & 3) | ((row >> 1) & 4)) << 1)) << 4);
}

// A chiplet's slot-th workgroup: the first tile of its group of rows (-1: it has none) and its
// run of columns, of `columns`. Tiles come in runs of one expert, a run's groups have four
// tiles, its last one maybe fewer. Uniform over a wave.
struct MoeSpot {
  int tile, column;
};
__device__ __forceinline__ MoeSpot moe_spot(const int* __restrict__ tile_expert, int n_tiles, int slot, int columns) {
  constexpr int PER = MOE_BM / MOE_MT;
  const int lane = threadIdx.x & (WAVE - 1), which = slot / columns;
  int seen = 0, run = 0;  // groups so far; first tile of the run that reaches into this chunk
  for (int base = 0; base < n_tiles; base += WAVE) {
    const int i = base + lane;
    const int e = i < n_tiles ? tile_expert[i] : -1;
    const int before = i > 0 && i <= n_tiles ? tile_expert[i - 1] : -1;
    const unsigned long long starts = __ballot(e != before || i == 0);
    const unsigned long long upto = starts & (~0ull >> (WAVE - 1 - lane));
    const int first = upto ? base + WAVE - 1 - __clzll((long long)upto) : run;
    const unsigned long long leads = __ballot(e >= 0 && ((i - first) & (PER - 1)) == 0);
    const int n = __popcll(leads);
    if (which < seen + n) {
      const bool mine = ((leads >> lane) & 1) && __popcll(leads & ((1ull << lane) - 1)) == which - seen;
      const int at = __ffsll((long long)__ballot(mine)) - 1;
      const int begin = __shfl(first, at), expert = __shfl(e, at);
      int end = base + at;
      for (unsigned long long same = ~0ull; same == ~0ull; end += same == ~0ull ? WAVE : __ffsll((long long)~same) - 1)
        same = __ballot(end + lane < n_tiles && tile_expert[min(end + lane, n_tiles - 1)] == expert);
      const int mid = (base + at - begin) / PER, chunk = mid & ~(MOE_SHARE - 1);
      const int share = min(MOE_SHARE, (end - begin + PER - 1) / PER - chunk);
      const int r = slot - columns * (which - mid + chunk);
      return {begin + PER * (chunk + r % share), r / share};
    }
    seen += n;
    if (starts) run = base + WAVE - 1 - __clzll((long long)starts);
  }
  return {-1, 0};
}

template <bool NF4>
__global__ __launch_bounds__(512, 2) void moe_gemm_kernel(
    const unsigned short* __restrict__ wt_all,      // [E, in, out] bf16 (NF4: null)
    const uint4* __restrict__ nf4_all,              // NF4: tiles (bf16: null)
    const unsigned short* __restrict__ scales_all,  // NF4: [E, out/64, n_kb * 128] bf16
    const unsigned short* __restrict__ x,           // [T, in] bf16
    const int* __restrict__ sorted_pairs,           // [Rp] pair id or -1 (padding)
    const int* __restrict__ tile_expert,            // [Rp/MT] expert id or -1
    unsigned short* __restrict__ c,                 // [R, out] bf16
    int in_dim,
    int out_dim,
    int k_per_tok,
    int n_tiles,
    int experts,
    int columns) {
  constexpr int BN = MOE_BN, BK = MOE_BK, T = 512;
  constexpr int AHEAD = NF4 ? 1 : 2;  // steps whose loads are in registers (NF4: codes last for two)
  constexpr int X_BYTES = MOE_BM * BK * 2, STAGE = X_BYTES + BN * BK * 2;
  extern __shared__ unsigned char smem[];
  __shared__ float2 lut2[NF4 ? 256 : 1];
  const MoeSpot spot = moe_spot(tile_expert, n_tiles, blockIdx.x >> 3, columns);
  const int tile = spot.tile, n0 = (spot.column * 8 + (blockIdx.x & 7)) * BN;
  if (tile < 0 || n0 >= out_dim) return;
  const int e = tile_expert[tile];
  if (e >= experts) return;
  int rows = MOE_MT;  // of this group
  while (rows < MOE_BM && tile + rows / MOE_MT < n_tiles && tile_expert[tile + rows / MOE_MT] == e) rows += MOE_MT;

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid & (WAVE - 1);
  const int col = lane & 15, hi = lane >> 4;
  const int wm = ((wave ^ (wave >> 2)) & 1) * 64, wn = wave / 2 * 64;  // this wave's rows and columns
  const bool idle = wm >= rows;                              // uniform over the wave
  if (NF4 && tid < 256) lut2[tid] = make_float2(MOE_NF4_LUT[tid & 0xF], MOE_NF4_LUT[tid >> 4]);

  // loads of a step: two 16-byte groups of X, and four of W, or for two steps two of NF4
  // codes (32 of a column) and for each step their 16 scales, per thread
  constexpr int X8 = BK / 8, XN = MOE_BM * X8 / T, WN = BK * BN / 8 / T;
  const unsigned short* xp[XN];
#pragma unroll
  for (int i = 0; i < XN; ++i) {
    const int row = (tid + i * T) / X8;
    const int pr = max(sorted_pairs[tile * MOE_MT + min(row, rows - 1)], 0);
    xp[i] = x + (size_t)(pr / k_per_tok) * in_dim + tid % X8 * 8;
  }
  const int wc = tid % (BN / 8) * 8, wr = tid / (BN / 8);  // first column and row of this thread's weights
  const unsigned short* wp =
      NF4 ? nullptr : wt_all + (size_t)e * in_dim * out_dim + (size_t)wr * out_dim + min(n0 + wc, out_dim - 8);
  const int n_kb = (in_dim + 127) / 128;

  short8 xn_all[AHEAD][XN], wn_all[AHEAD][NF4 ? 1 : WN];
  uint4 codes[2];
  short8 scale[2][2];
  auto fetch = [&](int step, short8* xn, short8* wnext) {
    const int kt = min(step, in_dim - BK);
#pragma unroll
    for (int i = 0; i < XN; ++i)
      xn[i] = *reinterpret_cast<const short8*>(xp[i] + kt);
    if constexpr (NF4) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int nb = min(n0 / 64 + tid / 256 + T / 256 * i, out_dim / 64 - 1);
        const size_t at = ((size_t)e * (out_dim / 64) + nb) * n_kb + kt / 128;
        if (step % 128 == 0) codes[i] = nf4_all[at * 256 + tid % 256];
        const short8* p = reinterpret_cast<const short8*>(scales_all + at * 128 + kt % 128 + lane / 16 * 16);
        scale[i][0] = p[0];
        scale[i][1] = p[1];
      }
    } else {
#pragma unroll
      for (int i = 0; i < WN; ++i)
        wnext[i] = *reinterpret_cast<const short8*>(wp + (size_t)(kt + i * 16) * out_dim);
    }
  };
  auto stage = [&](unsigned char* buf, int kt, const short8* xn, const short8* wnext) {
#pragma unroll
    for (int i = 0; i < XN; ++i) *reinterpret_cast<short8*>(buf + moe_x_at((tid + i * T) / X8, tid % X8)) = xn[i];
    unsigned char* w = buf + X_BYTES;
    if constexpr (NF4) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const unsigned words[2] = {kt & 64 ? codes[i].z : codes[i].x, kt & 64 ? codes[i].w : codes[i].y};
        const int row = (tid / 256 + T / 256 * i) * 64 + tid % 256 / 64 * 16 + col;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          short8 v;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const float2 two = lut2[(words[q] >> (8 * b)) & 0xFFu];
            v[b] = (short)f32_to_bf16(two.x * bf16_to_f32((unsigned short)scale[i][q][b]));
            v[b + 4] = (short)f32_to_bf16(two.y * bf16_to_f32((unsigned short)scale[i][q][b + 4]));
          }
          *reinterpret_cast<short8*>(w + moe_x_at(row, hi * 2 + q)) = v;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < WN; ++i) *reinterpret_cast<short8*>(w + moe_w_at(wr + i * 16, wc / 8)) = wnext[i];
    }
  };

  f32x4_moe acc[4][4];  // [columns][rows]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_moe{0.f, 0.f, 0.f, 0.f};
  static_assert(BK == 64);  // two halves of a step
  bf16x8_moe xf[2][4], wf[2][4];
  auto read = [&](const unsigned char* xb, int kc) {
    if (idle) return;
    const unsigned char* wb = xb + X_BYTES;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      xf[kc][j] = *reinterpret_cast<const bf16x8_moe*>(xb + moe_x_at(wm + j * 16 + col, kc * 4 + hi));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (NF4) {
        wf[kc][i] = *reinterpret_cast<const bf16x8_moe*>(wb + moe_x_at(wn + i * 16 + col, kc * 4 + hi));
      } else {
        // rows hi*8 + col/4 and 4 below, which are permuted alike; 4 columns a lane
        const int row = kc * 32 + hi * 8 + col / 4, group = (wn + i * 16) / 8 + ((col >> 1) & 1);
        wf[kc][i] = load_keys(reinterpret_cast<const unsigned short*>(wb + moe_w_at(row, group) + (col & 1) * 8), BN);
      }
    }
  };
  auto multiply = [&](int kc) {
    __builtin_amdgcn_sched_barrier(0);
    if (idle) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[kc][i], xf[kc][j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };

  // Step t lies in buffer t % 2; its loads are in registers t % AHEAD. A wave's step is two
  // intervals between barriers; waves 4 to 7, which have the same SIMDs as 0 to 3, are one
  // interval late. What an early wave writes in interval 2t, and a late one in 2t + 1, is
  // step t + 1's tile, read from 2t + 2 on; the buffer was last read in 2t - 1.
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) fetch(s * BK, xn_all[s], wn_all[s]);
  if (NF4) __syncthreads();  // the table
  stage(smem, 0, xn_all[0], wn_all[0]);
  __syncthreads();
  auto step = [&](int kt, int half) {
    constexpr int last = AHEAD - 1;
    read(smem + half * STAGE, 0);
    read(smem + half * STAGE, 1);
    stage(smem + (half ^ 1) * STAGE, kt + BK, xn_all[(half + 1) & last], wn_all[(half + 1) & last]);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    fetch(kt + (AHEAD + 1) * BK, xn_all[(half + 1) & last], wn_all[(half + 1) & last]);
    multiply(0);
    multiply(1);
    __syncthreads();
  };
  fetch(AHEAD * BK, xn_all[0], wn_all[0]);
  const bool late = wave >= 4;
  if (late) __syncthreads();
  int kt = 0;
  for (; kt + BK < in_dim; kt += 2 * BK) {
    step(kt, 0);
    step(kt + BK, 1);
  }
  if (kt < in_dim) {
    read(smem, 0);
    read(smem, 1);
    multiply(0);
    multiply(1);
  }
  if (!late) __syncthreads();

#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = wm + j * 16 + col;
    const int pr = row < rows ? sorted_pairs[tile * MOE_MT + row] : -1;
    if (pr < 0) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = n0 + wn + i * 16 + hi * 4;
      if (n < out_dim)
        *reinterpret_cast<v4s*>(c + (size_t)pr * out_dim + n) =
            v4s{(short)f32_to_bf16(acc[i][j][0]), (short)f32_to_bf16(acc[i][j][1]), (short)f32_to_bf16(acc[i][j][2]),
                (short)f32_to_bf16(acc[i][j][3])};
    }
  }
}

// bf16 weights, rows in groups of up to 256 that are as equal as tiles of 32 allow, by gemm_wide.h: two groups of 145
// rows are two tiles of 160 where groups of 128 rows were three, the last one nearly empty, and four waves take less
// from LDS for a product. Both products of a layer of 8 experts, width 4096 and inner size 14336, with 290 rows an expert
// and routing as it comes: from 698 and 405 to 571 and 310 us. With fewer rows weights are what bounds it (5.0 TB/s), and what it gains is that
// 128 columns keep more compute units busy: 10 rows an expert 318 and 318, 185 and 158 us. profiles/expert_products.csv has 1 to 750 rows:
// 1.5% slower at most, 14% faster in the mean.
struct MoeGroup {
  int tile, tiles, column;  // first tile and number of tiles (0: none); run of columns
};
// as moe_spot, with groups of up to `most` tiles
__device__ __forceinline__ MoeGroup moe_group_spot(const int* __restrict__ tile_expert, int n_tiles, int slot, int columns, int most) {
  const int lane = threadIdx.x & (WAVE - 1), which = slot / columns;
  int seen = 0, open = 0, open_expert = -1;  // groups so far; first tile of the run that is not closed yet, and whose
  for (int base = 0; base <= n_tiles; base += WAVE) {
    const int i = base + lane;
    const int e = i < n_tiles ? tile_expert[i] : -1;
    const int before = i > 0 && i <= n_tiles ? tile_expert[i - 1] : -1;
    const unsigned long long starts = __ballot(i <= n_tiles && (e != before || i == 0 || i == n_tiles));
    if (starts == 0) continue;
    // a run counts where it is closed: at the next one's start. Lane l has the run that ends at start l
    const bool closes = (starts >> lane) & 1;
    const unsigned long long below = starts & ((1ull << lane) - 1);
    const int from = below ? WAVE - 1 - __clzll((long long)below) : -1;
    const int run_expert = __shfl(e, max(from, 0));
    const int first = from >= 0 ? base + from : open, expert = from >= 0 ? run_expert : open_expert;
    const int length = closes && expert >= 0 ? i - first : 0, groups = (length + most - 1) / most;
    int upto = groups;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const int other = __shfl_up(upto, off);
      if (lane >= off) upto += other;
    }
    const unsigned long long here = __ballot(which < seen + upto);
    if (here) {
      const int at = __ffsll((long long)here) - 1;
      const int n = __shfl(groups, at), start = __shfl(first, at), size = __shfl(length, at), ahead = seen + __shfl(upto, at) - n;
      const int chunk = (which - ahead) & ~(MOE_SHARE - 1), share = min(MOE_SHARE, n - chunk);
      const int r = slot - columns * (ahead + chunk), group = chunk + r % share;
      const int each = size / n, more = size % n;  // the first `more` groups have one tile more
      return {start + group * each + min(group, more), each + (group < more), r / share};
    }
    seen += __shfl(upto, WAVE - 1);
    const int last = WAVE - 1 - __clzll((long long)starts);
    open = base + last;
    open_expert = __shfl(e, last);
  }
  return {-1, 0, 0};
}

// NARROW: 128 columns
template <int TILES, bool NARROW>
__device__ __forceinline__ void moe_wide_tile(
    unsigned char* lds, const unsigned short* w, const unsigned short* x, const int* pairs, unsigned short* c, int n0, int tokens,
    int in_dim, int out_dim, int k_per_tok) {
  constexpr int WR = NARROW || TILES > 5 ? 2 : 1, FM = 2 * TILES / WR, FN = NARROW ? 4 : 4 * WR;
  f32x4 acc[FN][FM];
  wide_product<false, WR, FM, FN>(
      lds, acc, wide_resource(x, (unsigned)tokens * in_dim * 2), wide_resource(w, (unsigned)in_dim * out_dim * 2),
      [&](int row) { return (unsigned)(max(pairs[row], 0) / k_per_tok) * in_dim * 2; },
      [&](int column) { return (unsigned)min(n0 + column, out_dim - 8); },
      (unsigned)out_dim * 2, 0, in_dim / MOE_BK);
  const int row = wide_row<false, WR, FM, FN>(), n = n0 + wide_column<false, WR, FM, FN>();
  int pr[FM];
#pragma unroll
  for (int j = 0; j < FM; ++j) pr[j] = pairs[row + j * 16];
  wide_store<FM, FN>(false, acc, [](auto) {}, [&](auto j, auto i, float (&v)[8], float (&)[8]) {
    if (pr[j] >= 0 && n + i * 32 < out_dim) store8(c + (size_t)pr[j] * out_dim + n + i * 32, v);
  });
}

template <bool NARROW>
__global__ __launch_bounds__(WIDE_THREADS, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void moe_wide_kernel(
    const unsigned short* __restrict__ wt_all, const unsigned short* __restrict__ x, const int* __restrict__ sorted_pairs,
    const int* __restrict__ tile_expert, unsigned short* __restrict__ c, int tokens, int in_dim, int out_dim, int k_per_tok, int n_tiles, int experts,
    int columns, int most) {
  extern __shared__ __align__(1024) unsigned char smem[];
  const MoeGroup spot = moe_group_spot(tile_expert, n_tiles, blockIdx.x >> 3, columns, most);
  const int tiles = __builtin_amdgcn_readfirstlane(spot.tiles), tile = __builtin_amdgcn_readfirstlane(spot.tile);
  const int n0 = __builtin_amdgcn_readfirstlane(spot.column * 8 + (blockIdx.x & 7)) * (NARROW ? 128 : 256);
  if (tiles == 0 || n0 >= out_dim) return;
  const int e = __builtin_amdgcn_readfirstlane(tile_expert[tile]);
  if (e >= experts) return;
  const unsigned short* w = wt_all + (size_t)e * in_dim * out_dim;
  const int* pairs = sorted_pairs + tile * MOE_MT;
#define MOE_TILES(N) \
  case N: moe_wide_tile<N, NARROW>(smem, w, x, pairs, c, n0, tokens, in_dim, out_dim, k_per_tok); break
  switch (tiles) {
    MOE_TILES(1);
    MOE_TILES(2);
    MOE_TILES(3);
    MOE_TILES(4);
  }
  if constexpr (!NARROW) switch (tiles) {
    MOE_TILES(5);
    MOE_TILES(6);
    MOE_TILES(7);
    MOE_TILES(8);
  }
#undef MOE_TILES
}

// ------------------------------------------------------------------- host

// x [T, dim] f32 or bf16, w [experts, dim] bf16 -> (weights [T, top] f32, experts [T, top] int32): the
// `top` largest of a softmax over all experts, renormalized
std::vector<torch::Tensor> moe_route(torch::Tensor x, torch::Tensor w, int64_t top) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() && w.is_cuda() && w.dtype() == torch::kBFloat16 &&
              w.dim() == 2 && w.is_contiguous() && w.size(1) == x.size(1));
  const long t = x.size(0), dim = x.size(1), experts = w.size(0);
  TORCH_CHECK(dim % 8 == 0 && top >= 1 && top <= experts && experts <= ROUTE_EXPERTS && top <= ROUTE_TOP);
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0);
  TORCH_CHECK(x.dtype() == torch::kFloat32 || x.dtype() == torch::kBFloat16);
  auto weights = torch::empty({t, top}, x.options().dtype(torch::kFloat32));
  auto sel = torch::empty({t, top}, x.options().dtype(torch::kInt32));
  if (t == 0) return {weights, sel};
  auto stream = at::cuda::getCurrentCUDAStream();
  if (x.dtype() == torch::kFloat32)
    moe_route_kernel<<<t, 256, 0, stream>>>(x.data_ptr<float>(), BF16P(w), weights.data_ptr<float>(),
                                            sel.data_ptr<int>(), (int)dim, (int)experts, (int)top);
  else
    moe_route_kernel<<<t, 256, 0, stream>>>((const unsigned short*)BF16P(x), BF16P(w), weights.data_ptr<float>(),
                                            sel.data_ptr<int>(), (int)dim, (int)experts, (int)top);
  HIP_CHECK_LAST();
  return {weights, sel};
}

// rows: partial sums [splits, T * top, out] f32, or [T * top, out] bf16 -> residual [T, out] + their weighted sum, bf16
torch::Tensor moe_combine(torch::Tensor rows, torch::Tensor weights, torch::Tensor residual) {
  TORCH_CHECK(weights.is_cuda() && weights.dtype() == torch::kFloat32 && weights.dim() == 2 && weights.is_contiguous());
  TORCH_CHECK(residual.is_cuda() && residual.dtype() == torch::kBFloat16 && residual.dim() == 2 && residual.is_contiguous());
  TORCH_CHECK(rows.is_cuda() && rows.is_contiguous());
  const long t = weights.size(0), top = weights.size(1), out_dim = residual.size(1);
  TORCH_CHECK(residual.size(0) == t && rows.size(-1) == out_dim && rows.size(-2) == t * top);
  auto y = torch::empty_like(residual);
  if (y.numel() == 0) return y;
  auto stream = at::cuda::getCurrentCUDAStream();
  if (rows.dim() == 3) {
    TORCH_CHECK(rows.dtype() == torch::kFloat32 && t <= 65535);
    moe_reduce_kernel<<<dim3((out_dim + 63) / 64, t), 1024, 0, stream>>>(
        rows.data_ptr<float>(), weights.data_ptr<float>(), BF16P(residual), BF16P(y), (int)rows.size(0), (int)t, (int)top,
        (int)out_dim);
  } else {
    TORCH_CHECK(rows.dim() == 2 && rows.dtype() == torch::kBFloat16 && out_dim % 8 == 0);
    TORCH_CHECK(reinterpret_cast<uintptr_t>(rows.data_ptr()) % 16 == 0 &&
                reinterpret_cast<uintptr_t>(residual.data_ptr()) % 16 == 0);
    const long groups = t * out_dim / 8, blocks = (groups + 255) / 256;
    TORCH_CHECK(blocks < (1L << 31));
    moe_combine_kernel<<<blocks, 256, 0, stream>>>(BF16P(rows), weights.data_ptr<float>(), BF16P(residual), BF16P(y),
                                                   (int)top, (int)out_dim, groups);
  }
  HIP_CHECK_LAST();
  return y;
}

// sel [R] expert of each (token, slot) pair -> (sorted_pairs, tile_expert) as moe_gemm takes them
std::vector<torch::Tensor> moe_group(torch::Tensor sel, int64_t experts, int64_t mt) {
  TORCH_CHECK(sel.is_cuda() && sel.dtype() == torch::kInt32 && sel.is_contiguous());
  TORCH_CHECK(experts >= 1 && experts <= 4096 && mt >= 1);
  const long r = sel.numel();
  // at most min(r, experts) segments end in a partly filled tile
  const long slots = (r + std::min(r, (long)experts) * (mt - 1) + mt - 1) / mt * mt;
  auto pairs = torch::empty({slots}, sel.options());
  auto tiles = torch::empty({slots / mt}, sel.options());
  moe_group_kernel<<<1, 1024, experts * 8, at::cuda::getCurrentCUDAStream()>>>(
      sel.data_ptr<int>(), r, experts, mt, slots, pairs.data_ptr<int>(), tiles.data_ptr<int>());
  HIP_CHECK_LAST();
  return {pairs, tiles};
}

// Most tiles of a group, 3 to 8: as many as possible, as a step of 64 of K takes about 0.35 us and 0.115 for each tile (what
// its weights take to come is shared by all), but with few columns a turn of all compute units is as long as its
// largest group. What routing gives is not known here: experts have 0.8 to 1.2 times the mean.
static int moe_most_tiles(long pairs, long experts, long columns) {
  int best = 8;
  float least = 0.f;
  for (int most = 8; most >= 3; --most) {
    float sum = 0.f, longest = 0.f;
    long units = 0;
    for (int i = 0; i < 5; ++i) {
      const long tiles = std::max(1L, (long)std::ceil((0.8f + 0.1f * i) * pairs / experts / MOE_MT));
      const long groups = (tiles + most - 1) / most, largest = (tiles + groups - 1) / groups;
      const float us = std::max(0.62f, 0.35f + 0.115f * largest);
      units += groups;
      sum += us * groups;
      longest = std::max(longest, us);
    }
    const float turns = (float)units * experts * columns / 5 / GEMM_CUS;
    const float us = turns < 4 ? std::ceil(turns) * longest : sum * experts * columns / 5 / GEMM_CUS + longest / 2;
    if (most == 8 || us < 0.99f * least) best = most, least = us;
  }
  return best;
}

static void launch_moe_wide(const torch::Tensor& wt_all, const torch::Tensor& x, const torch::Tensor& sorted_pairs,
                            const torch::Tensor& tile_expert, torch::Tensor& c, int64_t k_per_tok, int64_t n_rows) {
  const long experts = wt_all.size(0), in_dim = wt_all.size(1), out_dim = wt_all.size(2), n_tiles = tile_expert.size(0);
  if (n_tiles == 0 || x.size(0) == 0) return;
  // Few rows of few columns leave compute units without a tile of 256 columns, and weights are what is read: 8 experts of
  // 14336 x 4096 with 71 rows each, 218 us with 128 workgroups, 166 with 256.
  const long hit = std::min(experts, n_rows), mean = (long)std::ceil(1.2f * n_rows / experts / MOE_MT);
  const bool narrow = mean <= 4 && hit * ((out_dim + 255) / 256) <= GEMM_CUS * 5 / 8;
  const long bn = narrow ? 128 : 256, runs = (out_dim + bn - 1) / bn, columns = (runs + 7) / 8;
  const int most = narrow ? 4 : moe_most_tiles(n_rows, experts, runs);
  const long groups = std::min(n_tiles, (n_tiles + (most - 1) * experts) / most), blocks = groups * columns * 8;
  TORCH_CHECK(blocks < (1L << 31), "moe_gemm: too many rows");
#define MOE_WIDE(NARROW, LDS)                                                                                           \
  do {                                                                                                                  \
    const hipError_t fits = hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_wide_kernel<NARROW>),                \
                                                hipFuncAttributeMaxDynamicSharedMemorySize, LDS);                       \
    TORCH_CHECK(fits == hipSuccess, "moe_gemm: ", hipGetErrorString(fits));                                             \
    moe_wide_kernel<NARROW><<<blocks, WIDE_THREADS, LDS, at::cuda::getCurrentCUDAStream()>>>(                           \
        BF16P(wt_all), BF16P(x), sorted_pairs.data_ptr<int>(), tile_expert.data_ptr<int>(), BF16P(c), (int)x.size(0),          \
        (int)in_dim, (int)out_dim, (int)k_per_tok, (int)n_tiles, (int)experts, (int)columns, most);                     \
  } while (0)
  constexpr int WIDE_LDS = std::max(WideTile<false, 2, 8, 8>::LDS, WideTile<false, 1, 10, 4>::LDS);
  if (narrow) {
    constexpr int NARROW_LDS = WideTile<false, 2, 4, 4>::LDS;
    MOE_WIDE(true, NARROW_LDS);
  } else {
    MOE_WIDE(false, WIDE_LDS);
  }
#undef MOE_WIDE
  HIP_CHECK_LAST();
}

torch::Tensor moe_gemm(
    c10::optional<torch::Tensor> wt_all,      // [E, in, out] bf16
    c10::optional<torch::Tensor> nf4_all,     // NF4: [E, out/64, ceil(in/128), 4, 64, 16] u8
    c10::optional<torch::Tensor> scales_all,  // NF4: [E, out/64, ceil(in/128) * 128] bf16
    torch::Tensor x,                          // [T, in] bf16
    torch::Tensor sorted_pairs,               // [Rp] i32 (expert-sorted, MT-padded, -1 = pad)
    torch::Tensor tile_expert,                // [Rp/MT] i32 (-1 = pure padding tile)
    int64_t k_per_tok,
    int64_t n_rows,                           // R = T * k_per_tok (C rows)
    bool general) {                           // by moe_gemm_kernel whatever the sizes, for tests
  TORCH_CHECK(x.is_cuda() && x.dtype() == torch::kBFloat16 && x.dim() == 2 && x.is_contiguous());
  TORCH_CHECK(sorted_pairs.dtype() == torch::kInt32 && sorted_pairs.is_contiguous());
  TORCH_CHECK(tile_expert.dtype() == torch::kInt32 && tile_expert.is_contiguous());
  const bool nf4 = nf4_all.has_value();
  int in_dim, out_dim;
  if (nf4) {
    TORCH_CHECK(nf4_all->dtype() == torch::kUInt8 && nf4_all->dim() == 6 && nf4_all->is_contiguous());
    TORCH_CHECK(scales_all.has_value() && scales_all->dtype() == torch::kBFloat16 && scales_all->dim() == 3 &&
                scales_all->is_contiguous());
    in_dim = x.size(1);
    out_dim = nf4_all->size(1) * 64;
    TORCH_CHECK(nf4_all->size(2) == (in_dim + 127) / 128 && nf4_all->size(3) == 4 && nf4_all->size(4) == 64 &&
                nf4_all->size(5) == 16);
    TORCH_CHECK(scales_all->size(0) == nf4_all->size(0) && scales_all->size(1) == nf4_all->size(1) &&
                scales_all->size(2) == nf4_all->size(2) * 128);
  } else {
    TORCH_CHECK(wt_all.has_value() && wt_all->dtype() == torch::kBFloat16 && wt_all->dim() == 3 && wt_all->is_contiguous());
    in_dim = wt_all->size(1);
    out_dim = wt_all->size(2);
  }
  TORCH_CHECK(x.size(1) == in_dim);
  // staging loads are 16B/32-value vectors: callers fall back to the dense
  // path for geometries outside these alignments (fused_moe.py)
  TORCH_CHECK(out_dim % 128 == 0, "moe_gemm needs out_dim % 128 == 0");
  TORCH_CHECK(in_dim % 64 == 0, "moe_gemm needs in_dim % 64 == 0");
  const long Rp = sorted_pairs.size(0);
  TORCH_CHECK(Rp % MOE_MT == 0 && tile_expert.size(0) == Rp / MOE_MT);

  auto c = torch::empty({n_rows, (long)out_dim}, x.options());
  const long n_tiles = Rp / MOE_MT, experts = nf4 ? nf4_all->size(0) : wt_all->size(0);
  // offsets into an expert's weights and into rows are 32-bit there
  if (!general && !nf4 && (long)in_dim * out_dim < (1L << 31) && x.size(0) * in_dim < (1L << 31)) {
    launch_moe_wide(*wt_all, x, sorted_pairs, tile_expert, c, k_per_tok, n_rows);
    return c;
  }
  // an expert's last group may have one tile
  constexpr long per = MOE_BM / MOE_MT;
  const long groups = std::min(n_tiles, (n_tiles + (per - 1) * experts) / per);
  if (groups == 0 || x.size(0) == 0) return c;
  const long columns = (out_dim + 8 * MOE_BN - 1) / (8 * MOE_BN);  // runs of a chiplet
  const long blocks = groups * columns * 8;
  TORCH_CHECK(blocks < (1L << 31), "moe_gemm: too many rows");
  auto stream = at::cuda::getCurrentCUDAStream();
  const int lds = 2 * (MOE_BM + MOE_BN) * MOE_BK * 2;
#define MOE_GEMM(NF4, W, P, S)                                                                                   \
  do {                                                                                                           \
    const hipError_t fits = hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_gemm_kernel<NF4>),            \
                                                hipFuncAttributeMaxDynamicSharedMemorySize, lds);                \
    TORCH_CHECK(fits == hipSuccess, "moe_gemm: ", hipGetErrorString(fits));                                      \
    moe_gemm_kernel<NF4><<<blocks, 512, lds, stream>>>(                                                          \
        W, P, S, reinterpret_cast<const unsigned short*>(x.data_ptr()), sorted_pairs.data_ptr<int>(),            \
        tile_expert.data_ptr<int>(), reinterpret_cast<unsigned short*>(c.data_ptr()), in_dim, out_dim,           \
        (int)k_per_tok, (int)n_tiles, (int)experts, (int)columns);                                               \
  } while (0)
  if (nf4)
    MOE_GEMM(true, nullptr, reinterpret_cast<const uint4*>(nf4_all->data_ptr()),
             reinterpret_cast<const unsigned short*>(scales_all->data_ptr()));
  else
    MOE_GEMM(false, reinterpret_cast<const unsigned short*>(wt_all->data_ptr()), nullptr, nullptr);
#undef MOE_GEMM
  HIP_CHECK_LAST();
  return c;
}

torch::Tensor gemv_bf16_moe(
    torch::Tensor wt_all,    // [E, in, out] bf16
    torch::Tensor x,         // [B, in] f32
    torch::Tensor sel,       // [R] int32 (R = B * k)
    int64_t k_per_tok,
    torch::Tensor workspace,
    int64_t epilogue,
    int64_t splits_override,
    double limit,            // EPI_CLAMPED_SWIGLU_F32 only
    double alpha) {
  TORCH_CHECK(wt_all.is_cuda() && wt_all.dtype() == torch::kBFloat16 && wt_all.dim() == 3);
  TORCH_CHECK(x.dtype() == torch::kFloat32 && x.dim() == 2);
  TORCH_CHECK(sel.dtype() == torch::kInt32 && sel.is_contiguous());
  const int in_dim = wt_all.size(1), out_dim = wt_all.size(2);
  const int rows = sel.size(0);
  TORCH_CHECK(x.size(1) == in_dim && rows == x.size(0) * k_per_tok);
  TORCH_CHECK(rows <= 64, "moe gemv supports batch*k <= 64");
  if (splits_override <= 0 && gemv_mfma_fits(wt_all, out_dim)) {
    auto sums = launch_gemv_mfma(wt_all, x, &sel, k_per_tok, workspace);
    if (epilogue < 0) return sums;  // [splits, rows, out]
    return launch_gemv_reduce(
        sums, c10::nullopt, c10::nullopt, (int)sums.size(0), rows, out_dim, (int)epilogue, x.options(), wt_all.options(),
        c10::nullopt, ClampedGate{(float)limit, (float)alpha});
  }

  const long out_waves = (out_dim + GEMV_OUT_PER_WAVE - 1) / GEMV_OUT_PER_WAVE;
  long splits = splits_override > 0 ? splits_override : (768 + out_waves * rows - 1) / (out_waves * rows);
  long max_splits = (in_dim + 255) / 256;
  if (splits > max_splits) splits = max_splits;
  if (splits < 1) splits = 1;
  const int i_per_split = (in_dim + (int)splits - 1) / (int)splits;

  torch::Tensor partials;
  if (workspace.numel() >= (int64_t)splits * rows * out_dim) {
    partials = workspace;
  } else {
    partials = torch::empty({splits, (long)rows, (long)out_dim}, x.options());
  }
  dim3 grid(out_waves, splits, rows);
  auto stream = at::cuda::getCurrentCUDAStream();
  gemv_bf16_moe_kernel<<<grid, WAVE, 0, stream>>>(
      reinterpret_cast<const unsigned short*>(wt_all.data_ptr()), x.data_ptr<float>(),
      sel.data_ptr<int>(), partials.data_ptr<float>(), in_dim, out_dim, i_per_split,
      rows, (int)k_per_tok);
  HIP_CHECK_LAST();
  if (epilogue < 0) return partials.view(-1).narrow(0, 0, splits * rows * out_dim).view({splits, rows, out_dim});
  return launch_gemv_reduce(
      partials, c10::nullopt, c10::nullopt, (int)splits, rows, out_dim, (int)epilogue,
      x.options(), wt_all.options(), c10::nullopt, ClampedGate{(float)limit, (float)alpha});
}
