// Gradients of a prompt's causal attention for CDNA4 (gfx950): bf16 rows as the fused
// projection has them, grouped heads, rotated halves. From the rotated projection, the
// result, its rows' log2 of sums of weights and the result's gradient to the projection's
// gradient, turned back.
//
// Two kernels of one shape: a wave has 16 query rows (gradients of queries) or 16 keys
// (those of keys and values) as the columns of its products, and walks over tiles of 64 of
// the others, which four waves share in LDS, the next tile's loads in flight. Weights are
// made again from the scores, nothing of size rows x keys is ever in memory; weights and
// score gradients are the next product's operand without leaving their registers, as in
// paged_attn.h. Score gradients enter their products as three bf16 values, which hold all 24
// bits: products with 32-bit score gradients are what the results are to match. A workgroup
// of keys goes over all heads that share them.
//
// 32 heads of 128, 2 x 379 tokens: from the result's gradient back to the projection's it was
// 42 launches of torch operations over [heads, rows, keys] in 32 bits and over copies of
// rows, 419 us; the two kernels take 58 us, 29 and 29. (A row's mean taken from its rounded
// result and score gradients of 16 bits had saved 10 of 71.) Loads have no conditions, which
// would be branches between them, and a tile's sums and means come through LDS with its rows:
// the keys' kernel took 44 us with loads of a mean and a sum per score, in the midst of the
// products. At this size they are bound by the chain of a workgroup's tiles (six, and six times
// the heads that share keys): 384 workgroups for 256 compute units, 1.3 GFLOP of products.

#include "common.h"
#include "paged_attn.h"
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

#define AG_TILE 64  // rows of a tile

struct GradShape {
  int s, heads, kv_heads, start;
  long runs, sequences;
  float scale;
};

// 64 rows x HD of two matrices with the same rows -> LDS
template <int HD>
struct TilePair {
  static constexpr int ROW = HD + TPAD, D8 = HD / 8, NLD = AG_TILE * D8 / 256;
  bf16x8 a[NLD], b[NLD];
  // rows from j0 below s, zeros from there
  __device__ __forceinline__ void fetch(const unsigned short* pa, int sa, const unsigned short* pb, int sb, int j0, int s) {
    const auto ra = cached_rows(pa, j0, min(s - j0, AG_TILE), sa), rb = cached_rows(pb, j0, min(s - j0, AG_TILE), sb);
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int idx = threadIdx.x + i * 256, row = idx / D8, c = idx % D8 * 8;
      a[i] = load_cached(ra, (row * sa + c) * 2);
      b[i] = load_cached(rb, (row * sb + c) * 2);
    }
  }
  __device__ __forceinline__ void stage(unsigned short* buf) const {
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int idx = threadIdx.x + i * 256;
      unsigned short* dst = buf + idx / D8 * ROW + idx % D8 * 8;
      *reinterpret_cast<bf16x8*>(dst) = a[i];
      *reinterpret_cast<bf16x8*>(dst + AG_TILE * ROW) = b[i];
    }
  }
};

// [tile rows] x [this wave's 16 columns]
template <int HD>
__device__ __forceinline__ void tile_product(const unsigned short* lds, const bf16x8* frag, int col, int hi, f32x4* out) {
  constexpr int ROW = HD + TPAD;
#pragma unroll
  for (int nb = 0; nb < AG_TILE / 16; ++nb) {
    out[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < HD / 32; ++kc)
      out[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          *reinterpret_cast<const bf16x8*>(lds + (nb * 16 + col) * ROW + kc * 32 + hi * 8), frag[kc], out[nb], 0, 0, 0);
  }
}

// v = p[0] + p[1] + p[2], all its 24 bits
__device__ __forceinline__ void split_operand(const f32x4& a, const f32x4& b, bf16x8* p) {
  f32x4 ra = a, rb = b;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    p[i] = weight_operand(ra, rb);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ra[r] -= bf16_to_f32((unsigned short)p[i][r]);
      rb[r] -= bf16_to_f32((unsigned short)p[i][r + 4]);
    }
  }
}

// sums over a head's dims x 16 columns: a lane has one column and 4 neighbouring dims a block
template <int HD>
__device__ __forceinline__ void store_rotated(
    unsigned short* p, const f32x4* acc, float scale, const float* cos_t, const float* sin_t, int hi) {
  constexpr int HB = HD / 32;  // blocks of half a head
#pragma unroll
  for (int d = 0; d < HB; ++d) {
    const f32x4 c = *reinterpret_cast<const f32x4*>(cos_t + d * 16 + hi * 4);
    const f32x4 n = *reinterpret_cast<const f32x4*>(sin_t + d * 16 + hi * 4);
    v4s u, w;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float x = acc[d][r] * scale, y = acc[d + HB][r] * scale;
      u[r] = (short)f32_to_bf16(x * c[r] + y * n[r]);
      w[r] = (short)f32_to_bf16(y * c[r] - x * n[r]);
    }
    *reinterpret_cast<v4s*>(p + d * 16 + hi * 4) = u;
    *reinterpret_cast<v4s*>(p + HD / 2 + d * 16 + hi * 4) = w;
  }
}

// Gradients of queries, and `dots`: the mean by weight of each row's gradients of weights. It
// is what is taken off every one of them, so a walk of its own finds it in 32 bits first: the
// result times its gradient is the same number, but of a result that was rounded to bf16, and
// where keys are alike its error does not cancel (up to 0.5 of the terms that should have).
// Grid: runs of 64 rows x (batch, head) pairs.
template <int HD>
__global__ __launch_bounds__(256, 2) void attn_grad_q_kernel(
    const unsigned short* __restrict__ qkv,  // [B, S, (QH + 2 KH) HD], rotated
    const unsigned short* __restrict__ go,   // [B, S, QH HD]
    const float* __restrict__ lse,           // [B, QH, S], log2
    const float* __restrict__ cos_t, const float* __restrict__ sin_t,  // [positions, HD]
    unsigned short* __restrict__ grad,       // as qkv
    float* __restrict__ dots, GradShape a) { // [B, QH, S]
  constexpr int RC = HD / 32, VB = HD / 16, NB = AG_TILE / 16, ROW = HD + TPAD, BUF = 2 * AG_TILE * ROW;
  extern __shared__ unsigned short smem[];
  const int2 own = spread_tiles((int)a.runs, (int)a.sequences);
  const int b = own.y / a.heads, head = own.y % a.heads, kvh = head / (a.heads / a.kv_heads);
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid & (WAVE - 1), col = lane & 15, hi = lane >> 4;
  const int first = own.x * 64, r0 = first + wave * 16, row = r0 + col;
  const long width = (long)(a.heads + 2 * a.kv_heads) * HD, out_width = (long)a.heads * HD;
  const unsigned short* base = qkv + b * a.s * width;
  const unsigned short* kp = base + (a.heads + kvh) * HD;
  const unsigned short* vp = kp + a.kv_heads * HD;
  const bool live = row < a.s;
  // a lane without a row reads the last one: conditions would be branches between the loads
  const int safe = min(row, a.s - 1);
  const size_t at = ((size_t)b * a.s + safe) * out_width + head * HD, stat = ((size_t)b * a.heads + head) * a.s + safe;

  bf16x8 qf[RC], gf[RC];
#pragma unroll
  for (int kc = 0; kc < RC; ++kc) {
    qf[kc] = *reinterpret_cast<const bf16x8*>(base + safe * width + head * HD + kc * 32 + hi * 8);
    gf[kc] = *reinterpret_cast<const bf16x8*>(go + at + kc * 32 + hi * 8);
  }
  const float sum = lse[stat];
  f32x4 acc[VB];
#pragma unroll
  for (int d = 0; d < VB; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int key_end = min(a.s, first + 64), tiles = (key_end + AG_TILE - 1) / AG_TILE;
  const float in = a.scale * LOG2E;
  TilePair<HD> tile;
  auto fetch = [&](int step) { tile.fetch(kp, (int)width, vp, (int)width, step % tiles * AG_TILE, key_end); };
  fetch(0);
  tile.stage(smem);
  __syncthreads();
  auto walk = [&](int from, auto&& use) {  // over all tiles, the from-th step on
    for (int step = from; step < from + tiles; ++step) {
      const unsigned short* k_lds = smem + (step & 1) * BUF;
      const bool more = step + 1 < 2 * tiles;
      if (more) fetch(step + 1);
      f32x4 s[NB], ds[NB];
      tile_product<HD>(k_lds, qf, col, hi, s);
      tile_product<HD>(k_lds + AG_TILE * ROW, gf, col, hi, ds);
      const int j0 = (step - from) * AG_TILE + hi * 4;  // key of register 0 in block 0
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          s[nb][r] = live && j0 + nb * 16 + r <= row ? __builtin_amdgcn_exp2f(fmaf(s[nb][r], in, -sum)) : 0.f;
      use(k_lds, s, ds);
      if (more) tile.stage(smem + ((step + 1) & 1) * BUF);
      __syncthreads();
    }
  };
  float dot = 0.f, weight = 0.f;
  walk(0, [&](const unsigned short*, f32x4* s, f32x4* ds) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        weight += s[nb][r];
        dot = fmaf(s[nb][r], ds[nb][r], dot);
      }
  });
  weight = row_sum(weight);
  dot = row_sum(dot) / (live ? weight : 1.f);
  if (live && hi == 0) dots[stat] = dot;
  walk(tiles, [&](const unsigned short* k_lds, f32x4* s, f32x4* ds) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) ds[nb][r] = s[nb][r] * (ds[nb][r] - dot);
#pragma unroll
    for (int ks = 0; ks < NB / 2; ++ks) {
      bf16x8 parts[3];
      split_operand(ds[2 * ks], ds[2 * ks + 1], parts);
      const unsigned short* t = k_lds + (ks * 32 + hi * 4 + col / 4) * ROW + (col & 3) * 4;
#pragma unroll
      for (int d = 0; d < VB; ++d) {
        const bf16x8 kt = load_values(t + d * 16, ROW);
#pragma unroll
        for (int i = 2; i >= 0; --i) acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kt, parts[i], acc[d], 0, 0, 0);
      }
    }
  });
  if (live)
    store_rotated<HD>(grad + ((size_t)b * a.s + row) * width + head * HD, acc, a.scale, cos_t + (size_t)(a.start + row) * HD,
                      sin_t + (size_t)(a.start + row) * HD, hi);
}

// Gradients of keys and values. Grid: runs of 64 keys x (batch, head of keys) pairs.
template <int HD>
__global__ __launch_bounds__(256, 2) void attn_grad_kv_kernel(
    const unsigned short* __restrict__ qkv, const unsigned short* __restrict__ go, const float* __restrict__ lse,
    const float* __restrict__ dots, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
    unsigned short* __restrict__ grad, GradShape a) {
  constexpr int RC = HD / 32, VB = HD / 16, NB = AG_TILE / 16, ROW = HD + TPAD, BUF = 2 * AG_TILE * ROW;
  extern __shared__ unsigned short smem[];
  const int b = blockIdx.x / a.runs / a.kv_heads, kvh = blockIdx.x / a.runs % a.kv_heads, group = a.heads / a.kv_heads;
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid & (WAVE - 1), col = lane & 15, hi = lane >> 4;
  const int first = blockIdx.x % a.runs * 64, key = first + wave * 16 + col;  // early keys are seen most and come first
  const long width = (long)(a.heads + 2 * a.kv_heads) * HD, out_width = (long)a.heads * HD;
  const unsigned short* base = qkv + b * a.s * width;
  const bool live = key < a.s;

  bf16x8 kf[RC], vf[RC];
  const unsigned short* kp = base + min(key, a.s - 1) * width + (a.heads + kvh) * HD;
#pragma unroll
  for (int kc = 0; kc < RC; ++kc) {
    kf[kc] = *reinterpret_cast<const bf16x8*>(kp + kc * 32 + hi * 8);
    vf[kc] = *reinterpret_cast<const bf16x8*>(kp + a.kv_heads * HD + kc * 32 + hi * 8);
  }
  f32x4 dk[VB], dv[VB];
#pragma unroll
  for (int d = 0; d < VB; ++d) dk[d] = dv[d] = f32x4{0.f, 0.f, 0.f, 0.f};

  // steps: tiles of rows from `first` on, of one head after the other
  const int tiles = (a.s - first + AG_TILE - 1) / AG_TILE, steps = tiles * group;
  const float in = a.scale * LOG2E;
  TilePair<HD> tile;
  // with a tile's rows come their sums and means, 64 of each, which a lane needs 16 of
  float* const stats = reinterpret_cast<float*>(smem + 2 * BUF);
  const float* const mine = tid & 64 ? dots : lse;
  float stat;
  auto fetch = [&](int step) {
    const int head = kvh * group + step / tiles, j0 = first + step % tiles * AG_TILE;
    tile.fetch(base + head * HD, (int)width, go + (size_t)b * a.s * out_width + head * HD, (int)out_width, j0, a.s);
    stat = mine[((size_t)b * a.heads + head) * a.s + min(j0 + (tid & 63), a.s - 1)];
  };
  auto stage = [&](int which) {
    tile.stage(smem + which * BUF);
    if (tid < 2 * AG_TILE) stats[which * 2 * AG_TILE + tid] = stat;
  };
  fetch(0);
  stage(0);
  __syncthreads();
  for (int step = 0; step < steps; ++step) {
    const unsigned short* q_lds = smem + (step & 1) * BUF;
    const unsigned short* g_lds = q_lds + AG_TILE * ROW;
    const bool more = step + 1 < steps;
    if (more) fetch(step + 1);
    const int j0 = first + step % tiles * AG_TILE;
    f32x4 s[NB], ds[NB];
    tile_product<HD>(q_lds, kf, col, hi, s);
    tile_product<HD>(g_lds, vf, col, hi, ds);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const float* const of = stats + (step & 1) * 2 * AG_TILE + nb * 16 + hi * 4;
      const f32x4 sums = *reinterpret_cast<const f32x4*>(of), means = *reinterpret_cast<const f32x4*>(of + AG_TILE);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = j0 + nb * 16 + hi * 4 + r;
        const bool seen = live && row < a.s && key <= row;
        const float p = __builtin_amdgcn_exp2f(fmaf(s[nb][r], in, -sums[r]));
        s[nb][r] = seen ? p : 0.f;
        ds[nb][r] = seen ? p * (ds[nb][r] - means[r]) : 0.f;
      }
    }
#pragma unroll
    for (int ks = 0; ks < NB / 2; ++ks) {
      const bf16x8 pf = weight_operand(s[2 * ks], s[2 * ks + 1]);
      bf16x8 parts[3];
      split_operand(ds[2 * ks], ds[2 * ks + 1], parts);
      const int t = (ks * 32 + hi * 4 + col / 4) * ROW + (col & 3) * 4;
#pragma unroll
      for (int d = 0; d < VB; ++d) {
        dv[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_values(g_lds + t + d * 16, ROW), pf, dv[d], 0, 0, 0);
        const bf16x8 qt = load_values(q_lds + t + d * 16, ROW);
#pragma unroll
        for (int i = 2; i >= 0; --i) dk[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qt, parts[i], dk[d], 0, 0, 0);
      }
    }
    if (more) stage((step + 1) & 1);
    __syncthreads();
  }
  if (!live) return;
  unsigned short* p = grad + ((size_t)b * a.s + key) * width + (a.heads + kvh) * HD;
  store_rotated<HD>(p, dk, a.scale, cos_t + (size_t)(a.start + key) * HD, sin_t + (size_t)(a.start + key) * HD, hi);
#pragma unroll
  for (int d = 0; d < VB; ++d)
    *reinterpret_cast<v4s*>(p + a.kv_heads * HD + d * 16 + hi * 4) =
        v4s{(short)f32_to_bf16(dv[d][0]), (short)f32_to_bf16(dv[d][1]), (short)f32_to_bf16(dv[d][2]), (short)f32_to_bf16(dv[d][3])};
}

// -> the gradient of the projection before its rotation
torch::Tensor attn_prompt_grad(
    torch::Tensor qkv,  // [B, S, (qh + 2 kh) * hd] bf16, rotated
    torch::Tensor grad_out,  // [B, S, qh * hd] bf16
    torch::Tensor lse,  // [B, qh, S] f32
    torch::Tensor cos_t, torch::Tensor sin_t,  // [>= start + S, hd] f32
    int64_t start, int64_t qh, int64_t kh, int64_t hd, double scale) {
  TORCH_CHECK(hd == 64 || hd == 128, "gradients of attention support head_dim 64/128");
  TORCH_CHECK(qkv.is_cuda() && qkv.dim() == 3 && kh > 0 && qh > 0 && qh % kh == 0 && start >= 0);
  const long b = qkv.size(0), s = qkv.size(1);
  TORCH_CHECK(qkv.size(2) == (qh + 2 * kh) * hd);
  for (const auto* t : {&qkv, &grad_out})
    TORCH_CHECK(t->is_cuda() && t->dtype() == torch::kBFloat16 && t->is_contiguous() &&
                reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0, "contiguous bf16 rows, aligned to 16 bytes, expected");
  TORCH_CHECK(grad_out.dim() == 3 && grad_out.size(0) == b && grad_out.size(1) == s && grad_out.size(2) == qh * hd);
  TORCH_CHECK(lse.is_cuda() && lse.dtype() == torch::kFloat32 && lse.is_contiguous() && lse.numel() == b * qh * s);
  for (const auto* t : {&cos_t, &sin_t})
    TORCH_CHECK(t->is_cuda() && t->dtype() == torch::kFloat32 && t->is_contiguous() && t->dim() == 2 && t->size(1) == hd &&
                t->size(0) >= start + s && reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0, "rotation table too short");
  auto grad = torch::empty_like(qkv);
  if (b == 0 || s == 0) return grad;
  auto dots = torch::empty_like(lse);
  const long runs = (s + 63) / 64;
  // a tile's rows are addressed by 32 bits
  TORCH_CHECK(runs * b * qh < (1L << 31) && start + s < (1L << 31) && (qh + 2 * kh) * hd < (1L << 24), "too many rows at once");
  GradShape a{(int)s, (int)qh, (int)kh, (int)start, runs, b * qh, (float)scale};
  const size_t lds = 4 * AG_TILE * (hd + TPAD) * sizeof(unsigned short) + 4 * AG_TILE * sizeof(float);
  auto stream = at::cuda::getCurrentCUDAStream();
  auto bf = [](const torch::Tensor& t) { return reinterpret_cast<unsigned short*>(t.data_ptr()); };
#define ATTN_GRAD(HD)                                                                                               \
  do {                                                                                                              \
    allow_lds(&attn_grad_q_kernel<HD>, lds);                                                                        \
    allow_lds(&attn_grad_kv_kernel<HD>, lds);                                                                       \
    attn_grad_q_kernel<HD><<<runs * b * qh, 256, lds, stream>>>(                                                    \
        bf(qkv), bf(grad_out), lse.data_ptr<float>(), cos_t.data_ptr<float>(), sin_t.data_ptr<float>(),    \
        bf(grad), dots.data_ptr<float>(), a);                                                                       \
    attn_grad_kv_kernel<HD><<<runs * b * kh, 256, lds, stream>>>(                                                   \
        bf(qkv), bf(grad_out), lse.data_ptr<float>(), dots.data_ptr<float>(), cos_t.data_ptr<float>(),              \
        sin_t.data_ptr<float>(), bf(grad), a);                                                                      \
  } while (0)
  if (hd == 128)
    ATTN_GRAD(128);
  else
    ATTN_GRAD(64);
#undef ATTN_GRAD
  HIP_CHECK_LAST();
  return grad;
}
