// GQA decode attention for CDNA4 (gfx950), flash-decoding style.
//
// Default path (mfma_decode_kernel): scores as K Q^T and results as V^T P^T, the GQ query
// heads of one kv head (16 at a time) being the columns of both products, as in paged_attn.h:
// a lane has one head, its maximum takes two exchanges between lanes, and its weights are
// the second product's operand as they are. No tile passes through LDS: keys are read as
// operands, and of values a lane reads 8 (HD 64: 4) dims of the 8 keys whose weights it has
// and transposes them by byte permutes. Four waves take every fourth tile of 32 keys of
// their workgroup's part, with the next tile's loads in flight, and meet in LDS at the end;
// attn_decode_combine merges the parts.
//
// Bound by memory for long contexts, by two trips to it for short ones. MI355X, us with the
// combination, before (values through LDS, transposed one by one; every load waited for;
// weights through LDS) and now:
//   kv heads x queries each, head size, keys: 8 x 8, 128, 154           12.9 ->  6.2
//   8 x 8, 128, 2004                                                    18.8 ->  9.1
//   64 x 8, 128, 2004                                                   41.4 -> 18.9   3.5 TB/s
//   16 x 4, 128, 7901                                                   44.0 -> 18.0   3.6 TB/s
//   8 x 4, 128, 32000                                                   73.3 -> 32.7   4.0 TB/s
//   256 x 1, 128, 1000                                                  44.6 -> 25.3   5.2 TB/s
//   1 x 71, 64, 1000 (in cache)                                         39.8 -> 19.0
//
// The original VALU kernel (attn_decode_kernel: 16-lane-group dot products,
// online softmax in registers) is kept behind PETALS_DECODE_KERNEL=valu.
// kv_len comes from a DEVICE pointer so the whole decode step can be captured
// in a hipGraph with a moving position.
//
// Replaces the reference's torch QK^T/softmax/AV decode math
// (reference models/llama/block.py:108-127) on the MI355X fast path.

#include "common.h"
#include "paged_attn.h"
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

#include <cstdlib>

#define DKVT 32    // keys per wave-tile (MFMA path)
#define DWAVES 4   // waves per workgroup (MFMA path)

// Arbitrary GQ: heads are processed in ceil(GQ/16) groups of <=16 (one
// A-fragment each). The group loop sits OUTSIDE the kv loop so live registers
// stay at one group's footprint; K/V re-reads per extra group come from
// L2/HBM and are negligible for the weight-bound decode shapes that need
// GQ > 16 (falcon-7b MQA gq=71, falcon-180b gq=29 — reference
// models/falcon/block.py:100-110).
template <int HD, int GQ>
__global__ __launch_bounds__(DWAVES * 64, GQ > 16 ? 1 : 2) void mfma_decode_kernel(
    const float* __restrict__ q,            // [B, KV, GQ, HD]
    const unsigned short* __restrict__ k_cache,  // [B, KV, lmax, HD]
    const unsigned short* __restrict__ v_cache,
    float* __restrict__ part_o,             // [B*KV, splits, GQ, HD]
    float* __restrict__ part_ml,            // [B*KV, splits, GQ, 2]
    const int* __restrict__ kv_len_ptr,
    const float* __restrict__ alibi,        // [kv_heads*GQ] slopes or null
    int kv_heads,
    int lmax,
    int n_splits,
    float scale,
    float* __restrict__ out_direct) {  // n_splits==1: normalized out [B, KV*GQ*HD]
                                       // written here; the combine kernel is skipped
  constexpr int KC = HD / 32;
  constexpr int NV = HD / 16;                  // dims of a lane's values
  constexpr int GA = (GQ + 15) / 16;           // head groups of <=16
  constexpr int GN = GQ < 16 ? GQ : 16;
  constexpr int OROW = HD + 4;
  using values = __attribute__((ext_vector_type(NV / 2))) unsigned;
  using u32x4 = __attribute__((ext_vector_type(4))) unsigned;
  __shared__ float c_o[DWAVES][GN][OROW];
  __shared__ float c_ml[DWAVES][16][2];

  const int bkv = blockIdx.x;
  const int kvh = bkv % kv_heads;
  const int split = blockIdx.y;
  const int kv_len = *kv_len_ptr;
  const int rows_per_split = (kv_len + n_splits - 1) / n_splits;
  const int j_begin = split * rows_per_split;
  const int j_end = min(j_begin + rows_per_split, kv_len);

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid & (WAVE - 1);
  const int col = lane & 15, hi = lane >> 4;
  const size_t kv_base = (size_t)bkv * lmax * HD;
  const unsigned short* kb = k_cache + kv_base + hi * 8;
  const unsigned short* vb = v_cache + kv_base + col * NV;

  struct Tile {
    bf16x8 k[2][KC];  // keys col and 16 + col
    values v[8];      // keys hi*4 to +3 and 16 + hi*4 to +3
  };
  auto fetch = [&](Tile& t, int j0) {  // rows beyond the end repeat the last
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const unsigned short* row = kb + (size_t)min(j0 + nb * 16 + col, j_end - 1) * HD;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) t.k[nb][kc] = *reinterpret_cast<const bf16x8*>(row + kc * 32);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
      t.v[e] = *reinterpret_cast<const values*>(vb + (size_t)min(j0 + (e / 4) * 16 + hi * 4 + e % 4, j_end - 1) * HD);
  };

  for (int a = 0; a < GA; ++a) {
    const int g0 = a * 16;  // first head of this group
    // queries and the first tile, all on their way at once (queries one by one, each awaited, before the first tile:
    // 2 x 8 x 4 queries of 8000 keys 13.6 us, now 12.4)
    using f32x4_any = __attribute__((ext_vector_type(4), aligned(4))) float;
    f32x4 qv[KC][2];
    const float* qp = q + ((size_t)bkv * GQ + min(g0 + col, GQ - 1)) * HD + hi * 8;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc)
#pragma unroll
      for (int h = 0; h < 2; ++h) qv[kc][h] = *reinterpret_cast<const f32x4_any*>(qp + kc * 32 + h * 4);
    constexpr int STEP = DWAVES * DKVT;
    int j0 = j_begin + wave * DKVT;
    Tile one, two;
    if (j0 < j_end) fetch(one, j0);  // uniform over the wave
    bf16x8 qf[KC];
    const float q_scale = g0 + col < GQ ? scale : 0.f;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) qf[kc] = weight_operand(qv[kc][0] * q_scale, qv[kc][1] * q_scale);
    const float slope = alibi && g0 + col < GQ ? alibi[kvh * GQ + g0 + col] : 0.f;

    f32x4 acc[NV];  // [dim % NV][r]: dim (hi*4 + r) * NV + j of head g0 + col
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = NEG_SENTINEL, l = 0.f;  // l: this lane's share

    auto weigh = [&](Tile& t, int j0) {
      f32x4 s[2];
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        s[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) s[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t.k[nb][kc], qf[kc], s[nb], 0, 0, 0);
      }
      const int first = j0 + hi * 4;  // key of register 0 in block 0
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[nb][r] += slope * (first + nb * 16 + r);
      // masking and the maximum stay in separate loops (see prefill_attn.hip)
      if (j0 + DKVT > j_end) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (first + nb * 16 + r >= j_end) {
              s[nb][r] = NEG_SENTINEL;
              t.v[nb * 4 + r] = values{};
            }
      }
      float mx = m;
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[nb][r]);
      const float m_new = row_max(mx);
      if (__any(m_new > m)) {
        const float corr = m <= NEG_THRESHOLD ? 0.f : __expf(m - m_new);
        l *= corr;
        m = m_new;
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[j] *= corr;
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[nb][r] = s[nb][r] <= NEG_THRESHOLD ? 0.f : __expf(s[nb][r] - m);
          l += s[nb][r];
        }
      const bf16x8 p = weight_operand(s[0], s[1]);
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        u32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[i] = __builtin_amdgcn_perm(t.v[2 * i + 1][j / 2], t.v[2 * i][j / 2], j & 1 ? 0x07060302u : 0x05040100u);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, v), p, acc[j], 0, 0, 0);
      }
    };

    if (j0 < j_end) {
      for (;; j0 += 2 * STEP) {
        fetch(two, j0 + STEP);
        weigh(one, j0);
        if (j0 + STEP >= j_end) break;
        fetch(one, j0 + 2 * STEP);
        weigh(two, j0 + STEP);
        if (j0 + 2 * STEP >= j_end) break;
      }
    }

    // ---- cross-wave combine for this head group
    l = row_sum(l);
    if (a > 0) __syncthreads();  // the last group's sums have been read
    if (g0 + col < GQ) {
      float* dst = &c_o[wave][col][hi * 4 * NV];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < NV; j += 4)
          *reinterpret_cast<f32x4*>(dst + r * NV + j) = f32x4{acc[j][r], acc[j + 1][r], acc[j + 2][r], acc[j + 3][r]};
      if (hi == 0) {
        c_ml[wave][col][0] = m;
        c_ml[wave][col][1] = l;
      }
    }
    __syncthreads();

    const int gn = min(16, GQ - g0);  // heads in this group
    float* po = part_o + (((size_t)bkv * n_splits + split) * GQ + g0) * HD;
    float* pml = part_ml + (((size_t)bkv * n_splits + split) * GQ + g0) * 2;
    for (int idx = tid; idx < gn * HD; idx += DWAVES * WAVE) {
      const int gl = idx / HD, d = idx - gl * HD;
      float m_star = c_ml[0][gl][0];
#pragma unroll
      for (int w = 1; w < DWAVES; ++w) m_star = fmaxf(m_star, c_ml[w][gl][0]);
      float osum = 0.f, lsum = 0.f;
#pragma unroll
      for (int w = 0; w < DWAVES; ++w) {
        const float wgt = (c_ml[w][gl][0] <= NEG_THRESHOLD) ? 0.f : __expf(c_ml[w][gl][0] - m_star);
        osum += wgt * c_o[w][gl][d];
        lsum += wgt * c_ml[w][gl][1];
      }
      if (out_direct) {
        // single split: normalize here (matches the combine kernel's
        // n_splits==1 output exactly) and skip that kernel entirely
        out_direct[((size_t)bkv * GQ + g0 + gl) * HD + d] = osum / fmaxf(lsum, 1e-20f);
      } else {
        po[idx] = osum;
        if (d == 0) {
          pml[gl * 2 + 0] = m_star;
          pml[gl * 2 + 1] = lsum;
        }
      }
    }
  }
}

template <int HD, int GQ>
__global__ __launch_bounds__(64) void attn_decode_kernel(
    const float* __restrict__ q,           // [B, KV, GQ, HD]
    const unsigned short* __restrict__ k_cache,  // [Bc, KV, Lmax, HD]
    const unsigned short* __restrict__ v_cache,
    float* __restrict__ part_o,            // [B*KV, splits, GQ, HD]
    float* __restrict__ part_ml,           // [B*KV, splits, GQ, 2]
    const int* __restrict__ kv_len_ptr,
    const float* __restrict__ alibi,  // [kv_heads*GQ] slopes or null (ALiBi adds slope*j; the
                                      // row-constant part of the bias cancels in softmax)
    int kv_heads,
    int lmax,
    int n_splits,
    float scale) {
  constexpr int LANES_PER_ROW = 16;
  constexpr int EPL = HD / LANES_PER_ROW;  // elems per lane (8 for HD=128)
  constexpr int GROUPS = WAVE / LANES_PER_ROW;  // 4 rows in flight

  const int bkv = blockIdx.x;
  const int b = bkv / kv_heads;
  const int kv = bkv - b * kv_heads;
  const int split = blockIdx.y;
  const int kv_len = *kv_len_ptr;

  const int rows_per_split = (kv_len + n_splits - 1) / n_splits;
  const int j_begin = split * rows_per_split;
  const int j_end = min(j_begin + rows_per_split, kv_len);

  const int lane = threadIdx.x & (WAVE - 1);
  const int grp = lane / LANES_PER_ROW;  // 0..3
  const int gl = lane & (LANES_PER_ROW - 1);  // lane within group

  // stage q in LDS (scaled)
  __shared__ float q_lds[GQ][HD];
  for (int idx = threadIdx.x; idx < GQ * HD; idx += WAVE) {
    q_lds[idx / HD][idx % HD] = q[((size_t)(b * kv_heads + kv) * GQ) * HD + idx] * scale;
  }
  __syncthreads();

  float m[GQ], l[GQ], o[GQ][EPL];
#pragma unroll
  for (int g = 0; g < GQ; ++g) {
    m[g] = NEG_SENTINEL;
    l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) o[g][e] = 0.f;
  }

  const unsigned short* k_base = k_cache + ((size_t)b * kv_heads + kv) * lmax * HD;
  const unsigned short* v_base = v_cache + ((size_t)b * kv_heads + kv) * lmax * HD;

  float sl[GQ];
#pragma unroll
  for (int g = 0; g < GQ; ++g) sl[g] = alibi ? alibi[kv * GQ + g] : 0.f;

  for (int j = j_begin + grp; j < j_end; j += GROUPS) {
    // load K row slice: 16 lanes x EPL elems, coalesced
    const unsigned short* krow = k_base + (size_t)j * HD + gl * EPL;
    float kf[EPL];
    if (EPL == 8) {
      const short8 k8 = *reinterpret_cast<const short8*>(krow);
#pragma unroll
      for (int e = 0; e < 8; ++e) kf[e] = bf16_to_f32((unsigned short)k8[e]);
    } else {
#pragma unroll
      for (int e = 0; e < EPL; ++e) kf[e] = bf16_to_f32(krow[e]);
    }
    // scores for each q head of this group
    float s[GQ];
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
      float partial = 0.f;
#pragma unroll
      for (int e = 0; e < EPL; ++e) partial = fmaf(kf[e], q_lds[g][gl * EPL + e], partial);
      s[g] = group16_reduce_sum(partial) + sl[g] * j;  // all lanes get the row score
    }
    // V row slice
    const unsigned short* vrow = v_base + (size_t)j * HD + gl * EPL;
    float vf[EPL];
    if (EPL == 8) {
      const short8 v8 = *reinterpret_cast<const short8*>(vrow);
#pragma unroll
      for (int e = 0; e < 8; ++e) vf[e] = bf16_to_f32((unsigned short)v8[e]);
    } else {
#pragma unroll
      for (int e = 0; e < EPL; ++e) vf[e] = bf16_to_f32(vrow[e]);
    }
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
      const float m_new = fmaxf(m[g], s[g]);
      const float corr = __expf(m[g] - m_new);
      const float p = __expf(s[g] - m_new);
      l[g] = l[g] * corr + p;
#pragma unroll
      for (int e = 0; e < EPL; ++e) o[g][e] = o[g][e] * corr + p * vf[e];
      m[g] = m_new;
    }
  }

  // combine the 4 row-groups through LDS (deterministic order)
  __shared__ float c_m[GROUPS][GQ];
  __shared__ float c_l[GROUPS][GQ];
  __shared__ float c_o[GROUPS][GQ][HD];
  if (gl * EPL < HD) {
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) c_o[grp][g][gl * EPL + e] = o[g][e];
      if (gl == 0) {
        c_m[grp][g] = m[g];
        c_l[grp][g] = l[g];
      }
    }
  }
  __syncthreads();

  float* po = part_o + (((size_t)bkv * n_splits + split) * GQ) * HD;
  float* pml = part_ml + (((size_t)bkv * n_splits + split) * GQ) * 2;
  for (int idx = threadIdx.x; idx < GQ * HD; idx += WAVE) {
    const int g = idx / HD, d = idx % HD;
    float m_star = c_m[0][g];
#pragma unroll
    for (int r = 1; r < GROUPS; ++r) m_star = fmaxf(m_star, c_m[r][g]);
    float osum = 0.f, lsum = 0.f;
#pragma unroll
    for (int r = 0; r < GROUPS; ++r) {
      const float w = (c_m[r][g] <= NEG_THRESHOLD) ? 0.f : __expf(c_m[r][g] - m_star);
      osum += w * c_o[r][g][d];
      lsum += w * c_l[r][g];
    }
    po[idx] = osum;
    if (d == 0) {
      pml[g * 2 + 0] = m_star;
      pml[g * 2 + 1] = lsum;
    }
  }
}

// One workgroup per (batch and kv head, query head), of hd threads. The parts' weights are
// made once, then every thread's loads are independent.
__global__ void attn_decode_combine_kernel(
    const float* __restrict__ part_o,   // [B*KV, splits, GQ, HD]
    const float* __restrict__ part_ml,  // [B*KV, splits, GQ, 2]
    float* __restrict__ out,            // [B, KV*GQ*HD]
    int n_splits, int gq, int hd) {
  const int bkv = blockIdx.x;
  const int g = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  using f32x2 = __attribute__((ext_vector_type(2), aligned(4))) float;
  const f32x2* ml = reinterpret_cast<const f32x2*>(part_ml) + (size_t)bkv * n_splits * gq + g;
  const float* o = part_o + ((size_t)bkv * n_splits * gq + g) * hd + tid;
  // the first parts are asked for along with the maxima, and every wave weighs them by itself: one trip to memory
  // where there were three, and no barrier (16 parts: 7.0 us, now 4.7)
  constexpr int FIRST = 16;
  float part[FIRST];
#pragma unroll
  for (int i = 0; i < FIRST; ++i) part[i] = o[(size_t)min(i, n_splits - 1) * gq * hd];
  f32x2 v = lane < n_splits ? ml[(size_t)lane * gq] : f32x2{NEG_SENTINEL, 0.f};
  float m_star = v[0];
  for (int s = lane + WAVE; s < n_splits; s += WAVE) m_star = fmaxf(m_star, ml[(size_t)s * gq][0]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m_star = fmaxf(m_star, __shfl_xor(m_star, off, WAVE));
  float osum = 0.f, lsum = 0.f;
  for (int s0 = 0; s0 < n_splits; s0 += WAVE) {
    if (s0 > 0) v = s0 + lane < n_splits ? ml[(size_t)(s0 + lane) * gq] : f32x2{NEG_SENTINEL, 0.f};
    const float w = v[0] <= NEG_THRESHOLD ? 0.f : __expf(v[0] - m_star);
    lsum += wave_reduce_sum(w != 0.f ? w * v[1] : 0.f);
    auto weigh = [&](int i, float x) {
      const float wi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), i));
      osum += wi == 0.f ? 0.f : wi * x;
    };
    int i = 0;
    if (s0 == 0) {
#pragma unroll
      for (; i < FIRST; ++i) weigh(i, part[i]);  // no weight beyond the last
    }
    const int n = min(WAVE, n_splits - s0);
#pragma unroll 8
    for (; i < n; ++i) weigh(i, o[(size_t)(s0 + i) * gq * hd]);
  }
  out[((size_t)bkv * gq + g) * hd + tid] = osum / fmaxf(lsum, 1e-20f);
}

// ---------------------------------------------------------------- host API

// q: [B, KV*GQ*HD] f32 (token per row); caches [Bc, KV, Lmax, HD] bf16;
// kv_len: device int32 scalar tensor. Returns [B, KV*GQ*HD] f32.
torch::Tensor attn_decode_fused(
    torch::Tensor q,
    torch::Tensor k_cache,
    torch::Tensor v_cache,
    torch::Tensor kv_len,  // device int32 [1]
    int64_t gq,
    int64_t n_splits_i,
    torch::Tensor part_o,   // workspace [B*KV, splits, GQ, HD] f32 (or empty)
    torch::Tensor part_ml,  // workspace [B*KV, splits, GQ, 2] f32 (or empty)
    double scale,
    c10::optional<torch::Tensor> alibi_slopes) {  // [kv_heads*GQ] f32
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kFloat32);
  TORCH_CHECK(k_cache.dtype() == torch::kBFloat16 && k_cache.dim() == 4);
  const int b = q.size(0);
  const int kv_heads = k_cache.size(1), lmax = k_cache.size(2), hd = k_cache.size(3);
  const int GQi = (int)gq;
  static const bool use_valu = [] {
    const char* s = std::getenv("PETALS_DECODE_KERNEL");
    return s && s[0] == 'v';
  }();
  int n_splits = (int)n_splits_i;
  if (n_splits <= 0) {
    const int bkv = std::max(1, b * kv_heads);
    if (use_valu) {
      // VALU kernel: target ~1024 single-wave workgroups, chunks >= 64 rows
      n_splits = std::max(1, std::min(1024 / bkv, (lmax + 63) / 64));
    } else {
      // One workgroup for each of the 256 compute units, parts of 128 rows or more of a full
      // cache: two or three per unit were slower (32000 keys of 8 heads: 32 parts 31.7
      // us, 62 parts 39.6; 256 heads: 1 part 24.4, 2 parts 27.6). Up to 384 rows one
      // part, as the second launch costs more than the longer chain (300 keys of 8 heads: 8.1
      // us, 8.6 with 3 parts; of 32 heads 8.2, 8.7; 500 of 32 heads: 10.1, 8.8 with 4). Rows are those that the cache can
      // hold, as a captured launch stays while it fills; a short text in a long cache is read
      // in as many parts, of few rows each.
      static const int short_max = [] {
        const char* e = std::getenv("PETALS_AMD_DECODE_SHORT_LMAX");
        return e ? std::atoi(e) : 384;
      }();
      n_splits = lmax <= short_max ? 1 : std::max(1, std::min(256 / bkv, (lmax + 127) / 128));
    }
  }
  auto opts = q.options();
  const bool will_direct = !use_valu && n_splits == 1;  // parts go unused
  if (!will_direct && part_o.numel() < (int64_t)b * kv_heads * n_splits * GQi * hd)
    part_o = torch::empty({(int64_t)b * kv_heads, n_splits, GQi, hd}, opts);
  if (!will_direct && part_ml.numel() < (int64_t)b * kv_heads * n_splits * GQi * 2)
    part_ml = torch::empty({(int64_t)b * kv_heads, n_splits, GQi, 2}, opts);
  auto out = torch::empty({(int64_t)b, (int64_t)kv_heads * GQi * hd}, opts);

  dim3 grid(b * kv_heads, n_splits);
  auto stream = at::cuda::getCurrentCUDAStream();
  const float* qp = q.data_ptr<float>();
  const unsigned short* kp = reinterpret_cast<const unsigned short*>(k_cache.data_ptr());
  const unsigned short* vp = reinterpret_cast<const unsigned short*>(v_cache.data_ptr());
  float* pop = part_o.data_ptr<float>();
  float* pmlp = part_ml.data_ptr<float>();
  const int* lenp = kv_len.data_ptr<int>();
  const float sc = (float)scale;
  const float* alibi_p = nullptr;
  if (alibi_slopes.has_value() && alibi_slopes->defined() && alibi_slopes->numel() > 0) {
    TORCH_CHECK(alibi_slopes->is_contiguous() && alibi_slopes->dtype() == torch::kFloat32);
    TORCH_CHECK(alibi_slopes->numel() == (int64_t)kv_heads * GQi, "alibi slopes must be [q_heads]");
    alibi_p = alibi_slopes->data_ptr<float>();
  }

  // single split on the MFMA path: the decode kernel normalizes and writes
  // the output itself — the combine kernel (pure launch latency at short kv)
  // is skipped entirely
  float* direct_p = (!use_valu && n_splits == 1) ? out.data_ptr<float>() : nullptr;
  bool launched = false;
#define ATTN_CASE(HDV, GQV)                                                   \
  if (hd == HDV && GQi == GQV) {                                              \
    if (use_valu)                                                             \
      attn_decode_kernel<HDV, GQV><<<grid, 64, 0, stream>>>(                  \
          qp, kp, vp, pop, pmlp, lenp, alibi_p, kv_heads, lmax, n_splits, sc);\
    else                                                                      \
      mfma_decode_kernel<HDV, GQV><<<grid, DWAVES * WAVE, 0, stream>>>(       \
          qp, kp, vp, pop, pmlp, lenp, alibi_p, kv_heads, lmax, n_splits, sc, \
          direct_p);                                                          \
    launched = true;                                                          \
  }
  ATTN_CASE(128, 1) ATTN_CASE(128, 2) ATTN_CASE(128, 4) ATTN_CASE(128, 6)
  ATTN_CASE(128, 8) ATTN_CASE(128, 16)
  ATTN_CASE(64, 1) ATTN_CASE(64, 2) ATTN_CASE(64, 4) ATTN_CASE(64, 8) ATTN_CASE(64, 16)
#undef ATTN_CASE
  // GQ > 16 (multi-group MFMA path only; the VALU kernel would blow its
  // per-lane register arrays): falcon-7b MQA (gq=71), falcon-180b (gq=29)
#define ATTN_CASE_BIG(HDV, GQV)                                               \
  if (hd == HDV && GQi == GQV) {                                              \
    TORCH_CHECK(!use_valu, "VALU decode kernel does not support gq=", GQV);   \
    mfma_decode_kernel<HDV, GQV><<<grid, DWAVES * WAVE, 0, stream>>>(         \
        qp, kp, vp, pop, pmlp, lenp, alibi_p, kv_heads, lmax, n_splits, sc,   \
        direct_p);                                                            \
    launched = true;                                                          \
  }
  ATTN_CASE_BIG(64, 29) ATTN_CASE_BIG(64, 71) ATTN_CASE_BIG(64, 32)
  ATTN_CASE_BIG(128, 32)
#undef ATTN_CASE_BIG
  TORCH_CHECK(launched, "unsupported (head_dim, gqa) = (", hd, ", ", GQi, ")");
  HIP_CHECK_LAST();

  if (direct_p == nullptr) {
    dim3 cgrid(b * kv_heads, GQi);
    attn_decode_combine_kernel<<<cgrid, std::min(hd, 256), 0, stream>>>(
        pop, pmlp, out.data_ptr<float>(), n_splits, GQi, hd);
    HIP_CHECK_LAST();
  }
  return out;
}
