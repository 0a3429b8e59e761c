// RMS norms taken within the products that read them (decoding, few rows).
//
// The product of norm(h) = h * w / rms(h) is that of h * w, divided by rms(h) at the end: inputs are
// 16-bit products of two bf16 numbers, the factor of a row is known when the weights have arrived, and
// no launch of its own (2.9 us at width 2048, 4.5 us at 8192, as much as a small product) comes first.
// A row's sum of squares is either given in parts, by the kernel that wrote the row (gemv_reduce.h), or
// every workgroup sums the row up, which is 16 KB from L2 at width 8192: for few rows only. How few is
// ops/fused_decode.py's rule (norm_within), with times.
#pragma once

#include "common.h"
#include <torch/extension.h>

struct GemvNorm {
  const unsigned short* h;  // [rows, in] bf16
  const unsigned short* w;  // [in] bf16
  const float* sumsq;       // [rows, parts] or null
  int parts;
  float eps;
};

// by a workgroup of 4 waves: a wave's share of each row's sum of squares, to sq [4, rows] (LDS)
static __device__ __forceinline__ void norm_sums(const GemvNorm& n, int rows, int in_dim, float* sq) {
  const int tid = threadIdx.x;
  for (int r = 0; r < rows; ++r) {
    float s = 0.f;
    if (n.sumsq) {
      for (int i = tid; i < n.parts; i += 256) s += n.sumsq[(size_t)r * n.parts + i];
    } else {
      const unsigned short* row = n.h + (size_t)r * in_dim;
      for (int i = tid * 8; i < in_dim; i += 2048) {
        const short8 v = *reinterpret_cast<const short8*>(row + i);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float f = bf16_to_f32((unsigned short)v[j]);
          s = fmaf(f, f, s);
        }
      }
    }
    s = wave_reduce_sum(s);
    if ((tid & (WAVE - 1)) == 0) sq[tid / WAVE * rows + r] = s;
  }
}

static __device__ __forceinline__ float norm_factor(const GemvNorm& n, int rows, int r, int in_dim, const float* sq) {
  return rsqrtf(((sq[r] + sq[rows + r]) + (sq[2 * rows + r] + sq[3 * rows + r])) / in_dim + n.eps);
}

// A row's sum times its factor. Where the squares overflow (from 2^64 on they do) the factor is 0, and
// a norm of finite values is zeros, also where h * w or the sum is infinite; with an infinity among
// the row's values it is NaN, as that sum times 0. The bits are looked at: -ffast-math knows no
// infinities.
static __device__ __forceinline__ float norm_scaled(const GemvNorm& n, int rows, int r, int in_dim, const float* sq, float sum) {
  const float factor = norm_factor(n, rows, r, in_dim, sq);
  if (__float_as_uint(factor) == 0u) {
    bool finite = true;
    for (int i = 0; i < in_dim; ++i) finite &= (n.h[(size_t)r * in_dim + i] & 0x7FFF) < 0x7F80;
    if (finite) return 0.f;
  }
  return sum * factor;
}

// h [rows, in], w [in] and the sums of squares, as the kernels read them
static inline GemvNorm gemv_norm(const torch::Tensor& h, const torch::Tensor& w, const c10::optional<torch::Tensor>& sumsq,
                                 double eps) {
  TORCH_CHECK(h.is_cuda() && h.dtype() == torch::kBFloat16 && h.dim() == 2 && h.is_contiguous() && h.size(1) % 8 == 0);
  TORCH_CHECK(w.is_cuda() && w.dtype() == torch::kBFloat16 && w.dim() == 1 && w.is_contiguous() && w.size(0) == h.size(1));
  for (const auto& t : {h, w}) TORCH_CHECK(reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "rows are read 16 bytes at a time");
  GemvNorm n{reinterpret_cast<const unsigned short*>(h.data_ptr()), reinterpret_cast<const unsigned short*>(w.data_ptr()),
             nullptr, 0, (float)eps};
  if (sumsq.has_value()) {
    TORCH_CHECK(sumsq->is_cuda() && sumsq->dtype() == torch::kFloat32 && sumsq->dim() == 2 && sumsq->is_contiguous() &&
                sumsq->size(0) == h.size(0) && sumsq->size(1) > 0);
    n.sumsq = sumsq->data_ptr<float>();
    n.parts = (int)sumsq->size(1);
  }
  return n;
}
