// Shared device helpers for petals_amd CDNA4 (gfx950) kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#define WAVE 64

using short8 = __attribute__((ext_vector_type(8))) short;
using float4v = __attribute__((ext_vector_type(4))) float;

__device__ __forceinline__ float bf16_to_f32(unsigned short u) {
  union { float f; uint32_t i; } v;
  v.i = uint32_t(u) << 16;
  return v.f;
}

// to nearest, ties to even. One v_cvt_pk_bf16_f32, of two neighbouring values where both are needed, in the
// place of four whole-number operations a value
__device__ __forceinline__ unsigned short f32_to_bf16(float f) {
  return __builtin_bit_cast(unsigned short, (__bf16)f);
}

// GELU by its tanh form, 0.5 x (1 + tanh(u)) with u = sqrt(2 / pi) (x + 0.044715 x^3): x times the logistic function of 2u,
// from exp(-2|u|), which neither overflows nor takes numbers off each other that are nearly equal. Thirteen
// instructions where the library's tanh has two branches of some twenty: within a product's sums, where a wave
// has nobody to hide them, 513 us to 495 (4096 x 4096 x 16384). Error against 64 bits, relative in the 2-norm, here and by tanhf:
// 2.9e-8 and 3.1e-8 for normal values, 1.0e-7 and 3.8e-7 from -4 to -1, 5e-7 and 2e-3 below
__device__ __forceinline__ float gelu_tanh_f32(float x) {
  // -2 sqrt(2 / pi) log2(e), and 0.044715 times that
  const float t = __builtin_amdgcn_exp2f(-fabsf(x * fmaf(x * x, -0.10294324f, -2.3022082f))), d = 1.f + t;
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.f), r, r);
  const float q = t * r;
  return x > 0.f ? fmaf(-fminf(x, 1e30f), q, x) : x * q;
}

// full-wave fp32 sum (64 lanes)
__device__ __forceinline__ float wave_reduce_sum(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, WAVE);
  return x;
}

__device__ __forceinline__ float wave_reduce_max(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off, WAVE));
  return x;
}

// sum across a 16-lane subgroup (lanes with equal lane/16)
__device__ __forceinline__ float group16_reduce_sum(float x) {
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) x += __shfl_xor(x, off, WAVE);
  return x;
}

#define HIP_CHECK_LAST()                                                     \
  do {                                                                       \
    hipError_t e = hipGetLastError();                                        \
    if (e != hipSuccess) {                                                   \
      TORCH_CHECK(false, "HIP kernel launch failed: ", hipGetErrorString(e)); \
    }                                                                        \
  } while (0)

// finite stand-ins for -inf: the extension compiles with -ffast-math, under
// which IEEE inf comparisons/arithmetic are not reliable
#define NEG_SENTINEL  (-1e30f)
#define NEG_THRESHOLD (-1e29f)
