// Few rows times a bf16 matrix [in, out] on the matrix cores (gfx950).
//
// A wave has 128 columns and 32 S rows of the matrix, all of which it loads at once: lane l
// takes 8 columns, l%16, of the rows (l/16)*8 to +7 of each 32, which are four 64 x 16-byte
// loads away from an operand of v_mfma_f32_16x16x32_bf16: transposing the 8 x 8 values that
// a lane has is 32 byte permutes, and gives it eight inputs of one column for each of eight
// products. The other operand are the inputs, at most 8 rows of its 16 columns. They are
// 32-bit and stay so: x is the sum of three bf16 numbers (8 bits each, cut off rather than
// rounded), whose products are exact and summed in 32 bits.
//
// Unlike a product by vector operations, the cost does not grow with the rows, and the
// loads in flight do not shrink with the registers that more rows would take. Weights are
// read once and marked so (non-temporal: 43.5 instead of 47.0 us for the third line).
//
// Bound by memory: MI355X, us with the reduction, 1 and 8 rows; in brackets the kernel of
// gemv.hip with its own choice of splits, and with the best one that could be found:
//   2048 x 2048    6.4,  7.4   [ 25, 139;  17]
//   4096 x 6144   14.0, 16.8   [ 27, 151;  32 at 2 rows]
//   4096 x 28672  43.5, 55     [ 46, 189; 142 at 2 rows]   5.4 TB/s
//   14336 x 4096  25.7, 28     [ 34, 157;  60 at 2 rows]
// Error against 64 bits, of the root mean square result: 1.3e-7 [3.0e-7].
//
// With a norm's rows (gemv_norm.h), without the reduction: 2048 x 2560, 1 row, 5.4 us beside 7.2 with a norm
// ahead; 4096 x 6144, 2 rows, 12.7 beside 13.8.
#pragma once

#include "common.h"
#include "gemv_norm.h"
#include "paged.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>
#include <algorithm>

#define GEMV_MFMA_COLS 128

// x = p[0] + p[1] + p[2], eight values; infinities and NaNs in p[0] alone
static __device__ __forceinline__ void split_bf16(const float* x, bf16x8* p) {
  unsigned u[3][8], top = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    u[0][i] = __float_as_uint(x[i]);
    top = max(top, u[0][i] & 0x7FFFFFFFu);
    const float r = x[i] - __uint_as_float(u[0][i] & 0xFFFF0000u);
    u[1][i] = __float_as_uint(r);
    u[2][i] = __float_as_uint(r - __uint_as_float(u[1][i] & 0xFFFF0000u));
  }
  if (top >= 0x7F800000u) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if ((u[0][i] & 0x7FFFFFFFu) >= 0x7F800000u) {
        if (u[0][i] & 0x007FFFFFu) u[0][i] |= 0x00400000u;
        u[1][i] = u[2][i] = 0u;
      }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    using u32x4 = __attribute__((ext_vector_type(4))) unsigned;
    u32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_perm(u[q][2 * i + 1], u[q][2 * i], 0x07060302u);
    p[q] = __builtin_bit_cast(bf16x8, v);
  }
}

// Grid: (128 columns, runs of 4 x 32 S inputs, rows of sel or 1). With sel, there is one row,
// blockIdx.z: that of x[blockIdx.z / k_per_tok] with matrix sel[blockIdx.z].
// NORM: inputs are norm's rows instead of x (no sel).
template <int S, bool NORM>
static __global__ __launch_bounds__(256) void gemv_mfma_kernel(
    const unsigned short* __restrict__ wt,  // [in, out] or [experts, in, out]
    const float* __restrict__ x,            // [rows, in]
    const int* __restrict__ sel,            // [rows * k_per_tok] or null
    float* __restrict__ partials,           // [splits, rows or gridDim.z, out]
    int in_dim, int out_dim, int rows, int k_per_tok, int experts, bool by4, GemvNorm norm) {
  extern __shared__ float gemv_red[];  // [4 waves, rows, 128], and with NORM [4 waves, rows]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid & (WAVE - 1);
  const int col = lane & 15, hi = lane >> 4;
  const int n0 = blockIdx.x * GEMV_MFMA_COLS, k0 = (blockIdx.y * 4 + wave) * 32 * S;
  if (sel) {
    const int e = sel[blockIdx.z];
    if (e < 0 || e >= experts) return;  // uniform over the workgroup
    wt += (size_t)e * in_dim * out_dim;
    x += (size_t)(blockIdx.z / k_per_tok) * in_dim;
  }

  float xs[S][8];
  short8 hs[NORM ? S : 1], ws[NORM ? S : 1];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = k0 + s * 32 + hi * 8;
    const float* p = x + (size_t)col * in_dim + k;
    if constexpr (NORM) {  // in_dim is a multiple of 8; expanded when the weights are on their way
      hs[s] = ws[s] = short8{0, 0, 0, 0, 0, 0, 0, 0};
      if (col < rows && k < in_dim) {
        hs[s] = *reinterpret_cast<const short8*>(norm.h + (size_t)col * in_dim + k);
        ws[s] = *reinterpret_cast<const short8*>(norm.w + k);
      }
      continue;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) xs[s][i] = 0.f;
    if (col < rows) {
      if (by4 && k + 8 <= in_dim) {
        *reinterpret_cast<float4v*>(&xs[s][0]) = reinterpret_cast<const float4v*>(p)[0];
        *reinterpret_cast<float4v*>(&xs[s][4]) = reinterpret_cast<const float4v*>(p)[1];
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (k + i < in_dim) xs[s][i] = p[i];
      }
    }
  }
  using u32x4 = __attribute__((ext_vector_type(4))) unsigned;
  // columns beyond the matrix repeat its first ones; they are not stored
  const unsigned short* wp = wt + (size_t)(k0 + hi * 8) * out_dim + (n0 + col * 8 < out_dim ? n0 + col * 8 : n0);
  u32x4 w[S][8];
  if (k0 + 32 * S <= in_dim) {
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int r = 0; r < 8; ++r)
        w[s][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp + (size_t)(s * 32 + r) * out_dim));
  } else {
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        w[s][r] = u32x4{0u, 0u, 0u, 0u};
        if (k0 + hi * 8 + s * 32 + r < in_dim) w[s][r] = *reinterpret_cast<const u32x4*>(wp + (size_t)(s * 32 + r) * out_dim);
      }
  }
  __builtin_amdgcn_sched_barrier(0);
  float* sq = gemv_red + (size_t)4 * rows * GEMV_MFMA_COLS;
  if constexpr (NORM) norm_sums(norm, rows, in_dim, sq);

  f32x4 acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S; ++s) {
    bf16x8 xp[3], wf[8];
    if constexpr (NORM) {
#pragma unroll
      for (int i = 0; i < 8; ++i) xs[s][i] = bf16_to_f32((unsigned short)hs[s][i]) * bf16_to_f32((unsigned short)ws[s][i]);
    }
    split_bf16(xs[s], xp);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      u32x4 v;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        v[t] = __builtin_amdgcn_perm(w[s][2 * t + 1][j / 2], w[s][2 * t][j / 2], j & 1 ? 0x07060302u : 0x05040100u);
      wf[j] = __builtin_bit_cast(bf16x8, v);
    }
#pragma unroll
    for (int q = NORM ? 1 : 2; q >= 0; --q)  // 16 bits of a product are in two parts
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xp[q], acc[j], 0, 0, 0);
  }

  // acc[j][r]: row col, column (hi*4 + r)*8 + j
  if (col < rows) {
    float* dst = gemv_red + ((size_t)wave * rows + col) * GEMV_MFMA_COLS + hi * 32;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      *reinterpret_cast<float4v*>(dst + r * 8) = float4v{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
      *reinterpret_cast<float4v*>(dst + r * 8 + 4) = float4v{acc[4][r], acc[5][r], acc[6][r], acc[7][r]};
    }
  }
  __syncthreads();
  const int n = rows * GEMV_MFMA_COLS;
  for (int i = tid; i < n; i += 256) {
    const int c = n0 + i % GEMV_MFMA_COLS;
    if (c >= out_dim) continue;
    float sum = (gemv_red[i] + gemv_red[n + i]) + (gemv_red[2 * n + i] + gemv_red[3 * n + i]);
    if constexpr (NORM) sum = norm_scaled(norm, rows, i / GEMV_MFMA_COLS, in_dim, sq, sum);
    const size_t row = sel ? (size_t)blockIdx.y * gridDim.z + blockIdx.z : (size_t)blockIdx.y * rows + i / GEMV_MFMA_COLS;
    partials[row * out_dim + c] = sum;
  }
}

// rows of the matrix are read 16 bytes at a time
static bool gemv_mfma_fits(const torch::Tensor& wt, int64_t out_dim) {
  return out_dim % 8 == 0 && reinterpret_cast<uintptr_t>(wt.data_ptr()) % 16 == 0 && wt.is_contiguous();
}

// sel: [rows] matrices or null; with norm, x are the rows that it is of. Returns [splits, rows, out], f32
static torch::Tensor launch_gemv_mfma(
    const torch::Tensor& wt, const torch::Tensor& x, const torch::Tensor* sel, int64_t k_per_tok, torch::Tensor workspace,
    const GemvNorm* norm = nullptr) {
  const int lead = sel ? 1 : 0;
  const long in_dim = wt.size(lead), out_dim = wt.size(lead + 1);
  TORCH_CHECK(x.is_contiguous());
  const long rows = sel ? sel->numel() : x.size(0), z = sel ? rows : 1;
  const int batch = sel ? 1 : (int)x.size(0);
  const long columns = (out_dim + GEMV_MFMA_COLS - 1) / GEMV_MFMA_COLS;
  // two waves a SIMD, or as short as they get: 4096 x 4096 takes 10.8 us with 2048 waves of
  // 64 rows, 11.8 with 1024 of 128; from there on longer waves only save partial sums
  int s = 4;
  while (s > 1 && columns * z * ((in_dim + 32 * s - 1) / (32 * s)) < 2048) s /= 2;
  const long splits = std::max(1L, (in_dim + 128 * s - 1) / (128 * s));
  torch::Tensor partials = workspace.numel() >= splits * rows * out_dim
                               ? workspace.view(-1).narrow(0, 0, splits * rows * out_dim).view({splits, rows, out_dim})
                               : torch::empty({splits, rows, out_dim}, x.options().dtype(torch::kFloat32));
  if (rows == 0 || out_dim == 0) return partials;
  const bool by4 = in_dim % 4 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
  const dim3 grid(columns, splits, z);
  const size_t lds = sizeof(float) * 4 * batch * (GEMV_MFMA_COLS + (norm ? 1 : 0));
  auto stream = c10::hip::getCurrentHIPStream().stream();
#define GEMV_MFMA(S, NORM)                                                                                          \
  gemv_mfma_kernel<S, NORM><<<grid, 256, lds, stream>>>(                                                            \
      reinterpret_cast<const unsigned short*>(wt.data_ptr()), NORM ? nullptr : x.data_ptr<float>(),                 \
      sel ? sel->data_ptr<int>() : nullptr, partials.data_ptr<float>(), (int)in_dim, (int)out_dim, batch,           \
      (int)k_per_tok, sel ? (int)wt.size(0) : 1, by4, norm ? *norm : GemvNorm())
#define GEMV_MFMA_EITHER(S)             \
  do {                                  \
    if (norm) GEMV_MFMA(S, true);       \
    else GEMV_MFMA(S, false);           \
  } while (0)
  if (s == 4) GEMV_MFMA_EITHER(4);
  else if (s == 2) GEMV_MFMA_EITHER(2);
  else GEMV_MFMA_EITHER(1);
#undef GEMV_MFMA_EITHER
#undef GEMV_MFMA
  HIP_CHECK_LAST();
  return partials;
}
