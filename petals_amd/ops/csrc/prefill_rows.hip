// What stands between a prompt's dense products, one launch for each gap, bf16 rows:
//
//   qkv_rows        fused projection -> queries (in place), keys and values (to the cache or
//                   in place): bias, rotation of halves
//   add_norm_rows   residual + product (+ bias), and its RMS or layer norm
//   add_rows        x + y (+ z) (+ bias)
//   swiglu_rows     [rows, gate | up] -> silu(gate) * up
//   bias_gelu_rows  gelu(y + bias), in place
//
// and, where gradients are asked for, what stands between the products of the way back:
//
//   rotate_rows       qkv_rows to rows of their own
//   norm_rows_grad    gradient of an RMS norm's input (+ the residual's)
//   swiglu_rows_grad  gradient of [gate | up]
//
// All are bound by memory: every value is read and written once, 16 bytes at a time. As
// separate torch operations a llama block took 13 launches of about 5 us for them (and
// copies of queries, keys, gates and ups whose only purpose was their layout), which is
// what short prompts spent outside their products: 95 of 629 us at 128 tokens, width 8192.
// With gradients, a block's norms and gates were 59 launches, 404 us forward and back at
// 2 x 379 tokens, width 4096, inner size 11008; now 6, 50 us.

#include "common.h"
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

static __device__ __forceinline__ void load8f(const unsigned short* p, float* v) {
  const short8 a = *reinterpret_cast<const short8*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = bf16_to_f32((unsigned short)a[i]);
}
static __device__ __forceinline__ void store8f(unsigned short* p, const float* v) {
  short8 a;
#pragma unroll
  for (int i = 0; i < 8; ++i) a[i] = (short)f32_to_bf16(v[i]);
  *reinterpret_cast<short8*>(p) = a;
}

// A thread has 8 values of a head's first half and the 8 they turn into.
__global__ __launch_bounds__(256) void qkv_rows_kernel(
    const unsigned short* qkv,                // [B, S, (qh + 2 kh) * hd]
    unsigned short* out,                      // qkv, or the same elsewhere
    const unsigned short* __restrict__ bias,  // [(qh + 2 kh) * hd] or null
    const float* __restrict__ cos_t, const float* __restrict__ sin_t,  // [positions, hd] or null
    unsigned short* __restrict__ k_cache, unsigned short* __restrict__ v_cache,  // [B, kh, L, hd] or null
    long cache_batch, long cache_head, long cache_row, int s, int qh, int kh, int hd, int start, long units) {
  const long at = (long)blockIdx.x * 256 + threadIdx.x;
  if (at >= units) return;
  const int per_head = hd / 16, half = hd / 2;
  const int d = at % per_head * 8;
  const int head = at / per_head % (qh + 2 * kh);
  const long token = at / per_head / (qh + 2 * kh);
  const long b = token / s;
  const int i = token - b * s;
  const bool is_v = head >= qh + kh, turns = cos_t && !is_v;
  const unsigned short* p = qkv + (token * (qh + 2 * kh) + head) * hd + d;
  unsigned short* to = out + (p - qkv);
  if (k_cache && head >= qh)
    to = (is_v ? v_cache : k_cache) + b * cache_batch + (head - qh - (is_v ? kh : 0)) * cache_head + (start + i) * cache_row + d;
  if (to == p && !bias && !turns) return;
  float u[8], w[8];
  load8f(p, u);
  load8f(p + half, w);
  if (bias) {
    float c[8];
    load8f(bias + head * hd + d, c);
#pragma unroll
    for (int e = 0; e < 8; ++e) u[e] += c[e];
    load8f(bias + head * hd + d + half, c);
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] += c[e];
  }
  if (turns) {
    const float* c = cos_t + (size_t)(start + i) * hd + d;
    const float* n = sin_t + (size_t)(start + i) * hd + d;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = u[e], y = w[e];
      u[e] = x * c[e] - y * n[e];
      w[e] = y * c[e] + x * n[e];
    }
  }
  store8f(to, u);
  store8f(to + half, w);
}

#define NORM_KEEP 8  // groups of 8 values that a thread keeps between its passes: rows up to 16384

// h = x + y + y_bias; n = norm(h as stored). One row per workgroup.
template <bool LAYER>
__global__ __launch_bounds__(256) void add_norm_rows_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ y,
    const unsigned short* __restrict__ y_bias, const unsigned short* __restrict__ w,
    const unsigned short* __restrict__ b, unsigned short* __restrict__ h, unsigned short* __restrict__ n, int dim, float eps) {
  __shared__ float part[2][4];
  const size_t row = (size_t)blockIdx.x * dim;
  const int tid = threadIdx.x;
  float keep[NORM_KEEP][8], sum = 0.f, squares = 0.f;
#pragma unroll
  for (int i = 0; i < NORM_KEEP; ++i) {
    const int c = (tid + i * 256) * 8;
    if (c >= dim) continue;
    float t[8];
    load8f(x + row + c, keep[i]);
    load8f(y + row + c, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) keep[i][e] += t[e];
    if (y_bias) {
      load8f(y_bias + c, t);
#pragma unroll
      for (int e = 0; e < 8; ++e) keep[i][e] += t[e];
    }
    store8f(h + row + c, keep[i]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      keep[i][e] = bf16_to_f32(f32_to_bf16(keep[i][e]));
      sum += keep[i][e];
      squares = fmaf(keep[i][e], keep[i][e], squares);
    }
  }
  auto total = [&](float v, float* p) {
    v = wave_reduce_sum(v);
    if ((tid & 63) == 0) p[tid / 64] = v;
    __syncthreads();
    return (p[0] + p[1]) + (p[2] + p[3]);
  };
  float mean = 0.f, inv;
  if (LAYER) {
    mean = total(sum, part[0]) / dim;
    float dev = 0.f;  // squares about the mean
#pragma unroll
    for (int i = 0; i < NORM_KEEP; ++i)
      if ((tid + i * 256) * 8 < dim)
#pragma unroll
        for (int e = 0; e < 8; ++e) dev = fmaf(keep[i][e] - mean, keep[i][e] - mean, dev);
    inv = rsqrtf(total(dev, part[1]) / dim + eps);
  } else {
    inv = rsqrtf(total(squares, part[0]) / dim + eps);
  }
#pragma unroll
  for (int i = 0; i < NORM_KEEP; ++i) {
    const int c = (tid + i * 256) * 8;
    if (c >= dim) continue;
    float g[8];
    load8f(w + c, g);
#pragma unroll
    for (int e = 0; e < 8; ++e) keep[i][e] = (keep[i][e] - mean) * inv * g[e];
    if (LAYER) {
      load8f(b + c, g);
#pragma unroll
      for (int e = 0; e < 8; ++e) keep[i][e] += g[e];
    }
    store8f(n + row + c, keep[i]);
  }
}

// 8 values of a row per thread
__global__ __launch_bounds__(256) void add_rows_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ y, const unsigned short* __restrict__ z,
    const unsigned short* __restrict__ bias, unsigned short* __restrict__ out, int dim, long groups) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  if (g >= groups) return;
  float u[8], t[8];
  load8f(x + g * 8, u);
  load8f(y + g * 8, t);
#pragma unroll
  for (int e = 0; e < 8; ++e) u[e] += t[e];
  if (z) {
    load8f(z + g * 8, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) u[e] += t[e];
  }
  if (bias) {
    load8f(bias + g * 8 % dim, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) u[e] += t[e];
  }
  store8f(out + g * 8, u);
}

__global__ __launch_bounds__(256) void swiglu_rows_kernel(
    const unsigned short* __restrict__ gu, unsigned short* __restrict__ out, int inner, long groups) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  if (g >= groups) return;
  const long row = g * 8 / inner;
  const unsigned short* p = gu + row * 2 * inner + (g * 8 - row * inner);
  float a[8], u[8];
  load8f(p, a);
  load8f(p + inner, u);
#pragma unroll
  for (int e = 0; e < 8; ++e) a[e] = a[e] / (1.f + __expf(-a[e])) * u[e];
  store8f(out + g * 8, a);
}

// d/dx of sum(g * x / rms(x) * w), + residual; one row per workgroup
__global__ __launch_bounds__(256) void norm_rows_grad_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, const unsigned short* __restrict__ g,
    const unsigned short* __restrict__ residual, unsigned short* __restrict__ out, int dim, float eps) {
  __shared__ float part[2][4];
  const size_t row = (size_t)blockIdx.x * dim;
  const int tid = threadIdx.x;
  float keep[NORM_KEEP][8], turn[NORM_KEEP][8], squares = 0.f, dots = 0.f;
#pragma unroll
  for (int i = 0; i < NORM_KEEP; ++i) {
    const int c = (tid + i * 256) * 8;
    if (c >= dim) continue;
    float t[8];
    load8f(x + row + c, keep[i]);
    load8f(g + row + c, turn[i]);
    load8f(w + c, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      turn[i][e] *= t[e];
      squares = fmaf(keep[i][e], keep[i][e], squares);
      dots = fmaf(keep[i][e], turn[i][e], dots);
    }
  }
  squares = wave_reduce_sum(squares);
  dots = wave_reduce_sum(dots);
  if ((tid & 63) == 0) {
    part[0][tid / 64] = squares;
    part[1][tid / 64] = dots;
  }
  __syncthreads();
  squares = (part[0][0] + part[0][1]) + (part[0][2] + part[0][3]);
  dots = (part[1][0] + part[1][1]) + (part[1][2] + part[1][3]);
  const float inv = rsqrtf(squares / dim + eps), back = inv * inv * (dots / dim);
#pragma unroll
  for (int i = 0; i < NORM_KEEP; ++i) {
    const int c = (tid + i * 256) * 8;
    if (c >= dim) continue;
    float t[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (residual) load8f(residual + row + c, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] += inv * (turn[i][e] - keep[i][e] * back);
    store8f(out + row + c, t);
  }
}

__global__ __launch_bounds__(256) void swiglu_rows_grad_kernel(
    const unsigned short* __restrict__ gu, const unsigned short* __restrict__ g, unsigned short* __restrict__ out, int inner,
    long groups) {
  const long at = (long)blockIdx.x * 256 + threadIdx.x;
  if (at >= groups) return;
  const long row = at * 8 / inner, p = row * 2 * inner + (at * 8 - row * inner);
  float a[8], u[8], d[8];
  load8f(gu + p, a);
  load8f(gu + p + inner, u);
  load8f(g + at * 8, d);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float gate = 1.f / (1.f + __expf(-a[e])), silu = a[e] * gate;
    a[e] = d[e] * u[e] * gate * (1.f + a[e] * (1.f - gate));
    u[e] = d[e] * silu;
  }
  store8f(out + p, a);
  store8f(out + p + inner, u);
}

__global__ __launch_bounds__(256) void bias_gelu_rows_kernel(
    unsigned short* __restrict__ y, const unsigned short* __restrict__ bias, int dim, long groups) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  if (g >= groups) return;
  float v[8], c[8];
  load8f(y + g * 8, v);
  if (bias) {
    load8f(bias + g * 8 % dim, c);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += c[e];
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = gelu_tanh_f32(v[e]);
  store8f(y + g * 8, v);
}

// ------------------------------------------------------------------- host

#define U16(t) reinterpret_cast<unsigned short*>((t).data_ptr())

static void check_rows(const torch::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.dtype() == torch::kBFloat16 && t.is_contiguous(), "contiguous bf16 rows expected");
  TORCH_CHECK(t.dim() >= 1 && t.size(-1) % 8 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
              "rows must be multiples of 8 values, aligned to 16 bytes");
}

static const unsigned short* vector_or_null(const c10::optional<torch::Tensor>& t, int64_t n) {
  if (!t.has_value()) return nullptr;
  check_rows(*t);
  TORCH_CHECK(t->numel() == n);
  return U16(*t);
}

static long blocks_of(long threads) {
  TORCH_CHECK((threads + 255) / 256 < (1L << 31), "too many rows");
  return (threads + 255) / 256;
}

void qkv_rows(
    torch::Tensor qkv,  // [B, S, (qh + 2 kh) * hd]
    c10::optional<torch::Tensor> bias, c10::optional<torch::Tensor> cos_t, c10::optional<torch::Tensor> sin_t,
    c10::optional<torch::Tensor> k_cache, c10::optional<torch::Tensor> v_cache,  // [>= B, kh, L, hd]
    int64_t start, int64_t qh, int64_t kh, int64_t hd) {
  check_rows(qkv);
  TORCH_CHECK(qkv.dim() == 3 && hd % 16 == 0 && qh > 0 && kh > 0 && start >= 0 && qkv.size(2) == (qh + 2 * kh) * hd);
  const long b = qkv.size(0), s = qkv.size(1);
  const float *cp = nullptr, *sp = nullptr;
  if (cos_t.has_value()) {
    TORCH_CHECK(sin_t.has_value());
    for (const auto* t : {&*cos_t, &*sin_t})
      TORCH_CHECK(t->is_cuda() && t->dtype() == torch::kFloat32 && t->is_contiguous() && t->dim() == 2 &&
                  t->size(1) == hd && t->size(0) >= start + s, "rotation table too short");
    cp = cos_t->data_ptr<float>();
    sp = sin_t->data_ptr<float>();
  }
  unsigned short *kp = nullptr, *vp = nullptr;
  long cb = 0, ch = 0, cr = 0;
  if (k_cache.has_value()) {
    TORCH_CHECK(v_cache.has_value());
    for (const auto* t : {&*k_cache, &*v_cache}) {
      TORCH_CHECK(t->is_cuda() && t->dtype() == torch::kBFloat16 && t->dim() == 4 && t->strides() == k_cache->strides());
      TORCH_CHECK(t->stride(3) == 1 && t->stride(0) % 8 == 0 && t->stride(1) % 8 == 0 && t->stride(2) % 8 == 0 &&
                  reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0, "cache rows must be aligned to 16 bytes");
      TORCH_CHECK(t->size(0) >= b && t->size(1) == kh && t->size(3) == hd && t->size(2) >= start + s,
                  "the cache does not hold these rows");
    }
    kp = U16(*k_cache);
    vp = U16(*v_cache);
    cb = k_cache->stride(0);
    ch = k_cache->stride(1);
    cr = k_cache->stride(2);
  }
  const long units = b * s * (qh + 2 * kh) * (hd / 16);
  if (units == 0) return;
  qkv_rows_kernel<<<blocks_of(units), 256, 0, at::cuda::getCurrentCUDAStream()>>>(
      U16(qkv), U16(qkv), vector_or_null(bias, qkv.size(2)), cp, sp, kp, vp, cb, ch, cr, (int)s, (int)qh, (int)kh, (int)hd, (int)start,
      units);
  HIP_CHECK_LAST();
}

// the fused projection with queries and keys rotated
torch::Tensor rotate_rows(
    torch::Tensor qkv, torch::Tensor cos_t, torch::Tensor sin_t, int64_t start, int64_t qh, int64_t kh, int64_t hd) {
  check_rows(qkv);
  TORCH_CHECK(qkv.dim() == 3 && hd % 16 == 0 && qh > 0 && kh > 0 && start >= 0 && qkv.size(2) == (qh + 2 * kh) * hd);
  const long b = qkv.size(0), s = qkv.size(1);
  for (const auto* t : {&cos_t, &sin_t})
    TORCH_CHECK(t->is_cuda() && t->dtype() == torch::kFloat32 && t->is_contiguous() && t->dim() == 2 &&
                t->size(1) == hd && t->size(0) >= start + s, "rotation table too short");
  auto out = torch::empty_like(qkv);
  const long units = b * s * (qh + 2 * kh) * (hd / 16);
  if (units == 0) return out;
  qkv_rows_kernel<<<blocks_of(units), 256, 0, at::cuda::getCurrentCUDAStream()>>>(
      U16(qkv), U16(out), nullptr, cos_t.data_ptr<float>(), sin_t.data_ptr<float>(), nullptr, nullptr, 0, 0, 0, (int)s,
      (int)qh, (int)kh, (int)hd, (int)start, units);
  HIP_CHECK_LAST();
  return out;
}

// gradient of x, where g is that of its RMS norm with weight w, + residual
torch::Tensor norm_rows_grad(
    torch::Tensor x, torch::Tensor w, torch::Tensor g, c10::optional<torch::Tensor> residual, double eps) {
  check_rows(x);
  check_rows(g);
  const long dim = x.size(-1), rows = dim ? x.numel() / dim : 0;
  TORCH_CHECK(x.sizes() == g.sizes() && dim <= NORM_KEEP * 2048, "rows of up to 16384 values");
  if (residual.has_value()) {
    check_rows(*residual);
    TORCH_CHECK(residual->sizes() == x.sizes());
  }
  const unsigned short* wp = vector_or_null(w, dim);
  auto out = torch::empty_like(x);
  if (rows == 0) return out;
  TORCH_CHECK(rows < (1L << 31));
  norm_rows_grad_kernel<<<rows, 256, 0, at::cuda::getCurrentCUDAStream()>>>(
      U16(x), wp, U16(g), residual.has_value() ? U16(*residual) : nullptr, U16(out), (int)dim, (float)eps);
  HIP_CHECK_LAST();
  return out;
}

// gradient of [..., gate | up], where g is that of swiglu_rows
torch::Tensor swiglu_rows_grad(torch::Tensor gu, torch::Tensor g) {
  check_rows(gu);
  check_rows(g);
  TORCH_CHECK(gu.size(-1) == 2 * g.size(-1) && gu.numel() == 2 * g.numel());
  auto out = torch::empty_like(gu);
  const long groups = g.numel() / 8;
  if (groups == 0) return out;
  swiglu_rows_grad_kernel<<<blocks_of(groups), 256, 0, at::cuda::getCurrentCUDAStream()>>>(
      U16(gu), U16(g), U16(out), (int)g.size(-1), groups);
  HIP_CHECK_LAST();
  return out;
}

// -> (x + y + y_bias, its norm); b: of a layer norm, else an RMS norm
std::vector<torch::Tensor> add_norm_rows(
    torch::Tensor x, torch::Tensor y, c10::optional<torch::Tensor> y_bias, torch::Tensor w,
    c10::optional<torch::Tensor> b, double eps) {
  check_rows(x);
  check_rows(y);
  const long dim = x.size(-1), rows = dim ? x.numel() / dim : 0;
  TORCH_CHECK(x.sizes() == y.sizes() && dim <= NORM_KEEP * 2048, "rows of up to 16384 values");
  const unsigned short *yb = vector_or_null(y_bias, dim), *wp = vector_or_null(w, dim), *bp = vector_or_null(b, dim);
  auto h = torch::empty_like(x), n = torch::empty_like(x);
  if (rows == 0) return {h, n};
  TORCH_CHECK(rows < (1L << 31));
  auto stream = at::cuda::getCurrentCUDAStream();
  if (bp)
    add_norm_rows_kernel<true><<<rows, 256, 0, stream>>>(U16(x), U16(y), yb, wp, bp, U16(h), U16(n), (int)dim, (float)eps);
  else
    add_norm_rows_kernel<false><<<rows, 256, 0, stream>>>(U16(x), U16(y), yb, wp, bp, U16(h), U16(n), (int)dim, (float)eps);
  HIP_CHECK_LAST();
  return {h, n};
}

torch::Tensor add_rows(torch::Tensor x, torch::Tensor y, c10::optional<torch::Tensor> z, c10::optional<torch::Tensor> bias) {
  check_rows(x);
  check_rows(y);
  TORCH_CHECK(x.sizes() == y.sizes());
  if (z.has_value()) {
    check_rows(*z);
    TORCH_CHECK(z->sizes() == x.sizes());
  }
  const unsigned short* bp = vector_or_null(bias, x.size(-1));
  auto out = torch::empty_like(x);
  const long groups = x.numel() / 8;
  if (groups == 0) return out;
  add_rows_kernel<<<blocks_of(groups), 256, 0, at::cuda::getCurrentCUDAStream()>>>(
      U16(x), U16(y), z.has_value() ? U16(*z) : nullptr, bp, U16(out), (int)x.size(-1), groups);
  HIP_CHECK_LAST();
  return out;
}

// [..., gate | up] -> [..., inner]
torch::Tensor swiglu_rows(torch::Tensor gu) {
  check_rows(gu);
  TORCH_CHECK(gu.size(-1) % 16 == 0, "gates and ups must be multiples of 8 values");
  auto shape = gu.sizes().vec();
  shape.back() /= 2;
  auto out = torch::empty(shape, gu.options());
  const long groups = out.numel() / 8;
  if (groups == 0) return out;
  swiglu_rows_kernel<<<blocks_of(groups), 256, 0, at::cuda::getCurrentCUDAStream()>>>(
      U16(gu), U16(out), (int)shape.back(), groups);
  HIP_CHECK_LAST();
  return out;
}

void bias_gelu_rows(torch::Tensor y, c10::optional<torch::Tensor> bias) {
  check_rows(y);
  const unsigned short* bp = vector_or_null(bias, y.size(-1));
  const long groups = y.numel() / 8;
  if (groups == 0) return;
  bias_gelu_rows_kernel<<<blocks_of(groups), 256, 0, at::cuda::getCurrentCUDAStream()>>>(U16(y), bp, (int)y.size(-1), groups);
  HIP_CHECK_LAST();
}
