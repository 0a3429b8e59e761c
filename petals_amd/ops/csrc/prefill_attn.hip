// Flash attention of whole prompts over contiguous keys and values for CDNA4 (gfx950):
// bf16, causal or not, grouped heads, ALiBi. Queries, keys, values and results are read and
// written with the strides they have, so that a fused projection's rows serve as they are.
//
// The arithmetic of a tile is that of paged_attn.h: scores as K Q^T and results as V^T P^T,
// so that a lane has one query row, a row's maximum takes two exchanges between lanes, and
// weights are the next product's operand without leaving their registers. Four waves of 16
// or 32 rows of one head share double-buffered tiles of 64 keys; the next tile's loads are
// in flight during a tile's products. (The kernel before staged one tile at a time, wrote
// values to LDS transposed, one by one, and weights to LDS and back.)
//
// The loads of a tile are buffer loads, which give zeros beyond the last key, and a lane
// beyond the last row reads that one: with conditions each load was a branch of its own, and
// the loads waited for one another. Products have the priority of a SIMD's two waves: the
// other's softmax then runs beneath them.
//
// Bound by the products' operand loads from LDS and by the softmax's vector instructions,
// short ones by the chain of their tiles. MI355X, causal; loads under conditions, loads
// without, and with the products' priority:
//   64 heads of 128 over 8, 8192 tokens    1308   1255   1255 us   876 TFLOP/s
//   32 over 8, 4096 tokens                  186    181    181      759
//   32 over 8, 1024 tokens                 32.9   29.6   27.2
//   32 over 8, 512 tokens after 3584        113    109     98
//   32 over 8, 512 tokens                  18.5   16.7   15.4
//   71 heads of 64 over 1, 4 x 509 tokens    52     43     42
//   4 x 128 tokens, 32 heads of 128         8.3    7.5    7.1
// (The kernel that staged one tile at a time took 3534, 542, 266, 33.5 and 61 us for the
// sizes that it was measured at: the first, second, fourth, fifth and sixth.)
//
// NOTE: masking and the running maximum stay in separate loops (paged_attn.h
// weigh_tile). Fused (mask and `mx = fmaxf(mx, s)` in one loop body), amdclang (ROCm 7.2,
// gfx950, -O3, with or without -ffast-math) miscompiles the conditional sentinel store:
// dead keys keep their raw scores in register 0 of every accumulator row group
// (scripts/prefill_bisect.hip).
//
// Replaces the chunked rocBLAS-matmul + fp32-softmax prefill composition
// (ops/reference.py attention) on the GPU path; the reference framework used
// torch/CUDA attention inside HF blocks (reference models/llama/block.py:108).

#include "common.h"
#include "paged_attn.h"
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

#define PF_KEYS 64  // of a tile

// element strides; the last dimension is contiguous
struct Rows4 {
  const unsigned short* p;
  long batch, head, row;
};

// HD: head size, a multiple of 32; QB: blocks of 16 rows per wave.
// Grid: runs x sequences, runs of 64 QB rows, (batch, head) pairs as sequences.
template <int HD, int QB>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(
    Rows4 q, Rows4 k, Rows4 v, unsigned short* __restrict__ out, long out_batch, long out_head, long out_row,
    float* __restrict__ lse,  // [B, QH, S]: log2 of each row's sum of weights, or null
    AttnShape a, int runs, int sequences, int s_q, int kv_len, int kv_offset, bool causal) {
  constexpr int KT = PF_KEYS, NB = KT / 16, RC = HD / 32, VB = HD / 16;
  constexpr int ROW = HD + TPAD;        // of keys and of values in LDS
  constexpr int D8 = HD / 8;            // 16-byte groups of a row
  constexpr int NLD = KT * D8 / 256;    // per thread, of keys and of values
  extern __shared__ unsigned short smem[];

  const int2 own = spread_tiles(runs, sequences);
  const int b = own.y / a.heads, head = own.y % a.heads;
  const int kvh = head / (a.heads / a.kv_heads);
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid & (WAVE - 1);
  const int col = lane & 15, hi = lane >> 4;
  const int first = own.x * 64 * QB, r0 = first + wave * 16 * QB;
  const int last = min(first + 64 * QB, s_q) - 1;
  const int key_end = causal ? min(kv_len, kv_offset + last + 1) : kv_len;

  const ScoreScale scale = score_scale<SOFTMAX>(a);
  const float lin = linear_term<SOFTMAX>(a, head);
  const unsigned short* qp = q.p + b * q.batch + head * q.head;
  const unsigned short* kp = k.p + b * k.batch + kvh * k.head;
  const unsigned short* vp = v.p + b * v.batch + kvh * v.head;

  bf16x8 q_frag[QB][RC];
  f32x4 acc[QB][VB];
  float m[QB], l[QB];
  SeenRow seen[QB];
#pragma unroll
  for (int i = 0; i < QB; ++i) {
    const int row = r0 + i * 16 + col;
    const bool live = row < s_q;
    seen[i].pos = !live ? -1 : causal ? kv_offset + row : kv_len - 1;  // -1: sees nothing
    seen[i].lo = 0;
    m[i] = NEG_SENTINEL;
    l[i] = 0.f;
    // a lane without a row reads the last one: conditions would be branches between the loads
#pragma unroll
    for (int kc = 0; kc < RC; ++kc)
      q_frag[i][kc] = *reinterpret_cast<const bf16x8*>(qp + min(row, s_q - 1) * q.row + kc * 32 + hi * 8);
#pragma unroll
    for (int d = 0; d < VB; ++d) acc[i][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // keys that every row of this wave sees, and that some row sees: up to
  const int all_hi = r0 + 16 * QB > s_q ? -1 : causal ? kv_offset + r0 : kv_len - 1;
  const int any_hi = r0 >= s_q ? -1 : causal ? kv_offset + min(r0 + 16 * QB, s_q) - 1 : kv_len - 1;

  bf16x8 kn[NLD], vn[NLD];
  auto fetch = [&](int j0) {  // zeros beyond the last key
    const int rows = min(key_end - j0, KT), k_row = (int)k.row, v_row = (int)v.row;
    const auto kr = cached_rows(kp, j0, rows, k_row), vr = cached_rows(vp, j0, rows, v_row);
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int idx = tid + i * 256, row = idx / D8, c = idx % D8 * 8;
      kn[i] = load_cached(kr, (row * k_row + c) * 2);
      vn[i] = load_cached(vr, (row * v_row + c) * 2);
    }
  };
  auto stage = [&](unsigned short* buf) {
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int idx = tid + i * 256;
      unsigned short* dst = buf + idx / D8 * ROW + idx % D8 * 8;
      *reinterpret_cast<bf16x8*>(dst) = kn[i];
      *reinterpret_cast<bf16x8*>(dst + KT * ROW) = vn[i];
    }
  };

  fetch(0);
  stage(smem);
  __syncthreads();
  int which = 0;
  for (int j0 = 0; j0 < key_end; j0 += KT, which ^= 1) {
    const unsigned short* k_lds = smem + which * 2 * KT * ROW;
    const bool more = j0 + KT < key_end;
    if (more) fetch(j0 + KT);
    if (j0 <= any_hi) {  // uniform over the wave
      const bool interior = j0 + KT - 1 <= all_hi && j0 + KT <= key_end;
      bf16x8 p_frag[QB][NB / 2];
      f32x4 s[QB][NB];
      __builtin_amdgcn_s_setprio(1);  // see above
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int i = 0; i < QB; ++i) s[i][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < RC; ++kc) {
          const bf16x8 kt = *reinterpret_cast<const bf16x8*>(&k_lds[(nb * 16 + col) * ROW + kc * 32 + hi * 8]);
#pragma unroll
          for (int i = 0; i < QB; ++i) s[i][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kt, q_frag[i][kc], s[i][nb], 0, 0, 0);
        }
      }
      __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int i = 0; i < QB; ++i) {
        float corr;
        if (weigh_tile<SOFTMAX, NB>(s[i], m[i], l[i], lin, seen[i], j0, hi, key_end, interior, scale, corr)) {
#pragma unroll
          for (int d = 0; d < VB; ++d) acc[i][d] *= corr;
        }
#pragma unroll
        for (int ks = 0; ks < NB / 2; ++ks) p_frag[i][ks] = weight_operand(s[i][2 * ks], s[i][2 * ks + 1]);
      }
      const unsigned short* v_lds = k_lds + KT * ROW + (hi * 4 + col / 4) * ROW + (col & 3) * 4;
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int d = 0; d < VB; ++d)
#pragma unroll
        for (int ks = 0; ks < NB / 2; ++ks) {
          const bf16x8 vt = load_values(v_lds + ks * 32 * ROW + d * 16, ROW);
#pragma unroll
          for (int i = 0; i < QB; ++i) acc[i][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt, p_frag[i][ks], acc[i][d], 0, 0, 0);
        }
      __builtin_amdgcn_s_setprio(0);
    }
    if (more) stage(smem + (which ^ 1) * 2 * KT * ROW);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < QB; ++i) {
    const int row = r0 + i * 16 + col;
    const float sum = row_sum(l[i]), inv = sum > 0.f ? 1.f / sum : 0.f;
    if (row >= s_q) continue;
    if (lse && hi == 0) lse[(size_t)own.y * s_q + row] = m[i] + log2f(sum);
    unsigned short* dst = out + b * out_batch + head * out_head + row * out_row + hi * 4;
#pragma unroll
    for (int d = 0; d < VB; ++d)
      *reinterpret_cast<v4s*>(dst + d * 16) =
          v4s{(short)f32_to_bf16(acc[i][d][0] * inv), (short)f32_to_bf16(acc[i][d][1] * inv),
              (short)f32_to_bf16(acc[i][d][2] * inv), (short)f32_to_bf16(acc[i][d][3] * inv)};
  }
}

// rows that 16-byte loads can read as they lie, one after the other and within 32 bits for a tile, else a copy
static torch::Tensor readable_rows(const torch::Tensor& t) {
  bool ok = t.stride(3) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  ok = ok && t.stride(2) >= t.size(3) && t.stride(2) < (1L << 24);
  for (int i = 0; i < 3; ++i) ok = ok && (t.size(i) == 1 || t.stride(i) % 8 == 0);
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

static Rows4 rows4(const torch::Tensor& t) {
  return Rows4{reinterpret_cast<const unsigned short*>(t.data_ptr()), t.stride(0), t.stride(1), t.stride(2)};
}

// q [B, QH, S, HD], k and v [B, KVH, Lmax, HD] of any strides; out likewise, rows aligned to 8 bytes
static void run_prefill(
    torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor out, int64_t kv_len, int64_t kv_offset, double scale,
    bool causal, const c10::optional<torch::Tensor>& alibi_slopes, float* lse = nullptr) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16 && q.dim() == 4);
  TORCH_CHECK(k.dtype() == torch::kBFloat16 && k.dim() == 4 && v.dtype() == torch::kBFloat16 && v.dim() == 4);
  const int B = q.size(0), QH = q.size(1), S = q.size(2), HD = q.size(3);
  const int KVH = k.size(1);
  TORCH_CHECK(HD == 128 || HD == 64, "prefill attention supports head_dim 64/128");
  TORCH_CHECK(QH % KVH == 0);
  TORCH_CHECK(k.size(0) >= B && v.size(0) >= B && v.size(1) == KVH && k.size(3) == HD && v.size(3) == HD);
  TORCH_CHECK(kv_len >= 0 && kv_len <= k.size(2) && kv_len <= v.size(2), "more keys than the cache holds");
  AttnShape a{};
  a.heads = QH;
  a.kv_heads = KVH;
  a.scale = (float)scale;
  if (alibi_slopes.has_value() && alibi_slopes->defined() && alibi_slopes->numel() > 0) {
    TORCH_CHECK(alibi_slopes->is_contiguous() && alibi_slopes->dtype() == torch::kFloat32);
    TORCH_CHECK(alibi_slopes->numel() == QH, "alibi slopes must be [q_heads]");
    a.slopes = alibi_slopes->data_ptr<float>();
  }
  if (B == 0 || S == 0) return;
  q = readable_rows(q);
  k = readable_rows(k);
  v = readable_rows(v);
  // 32 rows a wave halve the loads of keys and values per product, as long as that leaves two
  // workgroups for each compute unit
  const bool wide = (long)B * QH * ((S + 127) / 128) >= 512;
  const long runs = (S + (wide ? 127 : 63)) / (wide ? 128 : 64), sequences = (long)B * QH;
  TORCH_CHECK(runs * sequences < (1L << 31), "too many rows at once");
  const size_t lds = 4 * PF_KEYS * (HD + TPAD) * sizeof(unsigned short);
  auto stream = at::cuda::getCurrentCUDAStream();
#define PREFILL(HDV, QB)                                                                                              \
  do {                                                                                                                \
    allow_lds(&attn_prefill_kernel<HDV, QB>, lds);                                                                    \
    attn_prefill_kernel<HDV, QB><<<runs * sequences, 256, lds, stream>>>(                                                         \
        rows4(q), rows4(k), rows4(v), reinterpret_cast<unsigned short*>(out.data_ptr()), out.stride(0), out.stride(1), \
        out.stride(2), lse, a, (int)runs, (int)sequences, S, (int)kv_len, (int)kv_offset, causal);                         \
  } while (0)
  if (HD == 128) {
    if (wide) PREFILL(128, 2);
    else PREFILL(128, 1);
  } else {
    if (wide) PREFILL(64, 2);
    else PREFILL(64, 1);
  }
#undef PREFILL
  HIP_CHECK_LAST();
}

torch::Tensor attn_prefill_fused(
    torch::Tensor q,  // [B, QH, S, HD] bf16
    torch::Tensor k,  // [B, KVH, Lmax, HD] bf16 (cache; valid prefix kv_len)
    torch::Tensor v,
    int64_t kv_len,
    int64_t kv_offset,
    double scale,
    bool causal,
    c10::optional<torch::Tensor> alibi_slopes) {  // [QH] f32
  TORCH_CHECK(q.is_contiguous() && k.is_contiguous() && v.is_contiguous());
  auto out = torch::empty(q.sizes(), q.options());
  run_prefill(q, k, v, out, kv_len, kv_offset, scale, causal, alibi_slopes);
  return out;
}

// the same with results as rows of tokens: [B, S, QH * HD]
torch::Tensor attn_prefill_rows(
    torch::Tensor q, torch::Tensor k, torch::Tensor v, int64_t kv_len, int64_t kv_offset, double scale, bool causal,
    c10::optional<torch::Tensor> alibi_slopes) {
  TORCH_CHECK(q.dim() == 4);
  auto out = torch::empty({q.size(0), q.size(2), q.size(1) * q.size(3)}, q.options());
  run_prefill(q, k, v, out.view({q.size(0), q.size(2), q.size(1), q.size(3)}).transpose(1, 2), kv_len, kv_offset, scale,
              causal, alibi_slopes);
  return out;
}

// what training keeps: a prompt's causal attention over itself, and [B, QH, S] log2 of the sums of its rows' weights
std::vector<torch::Tensor> attn_prefill_sums(torch::Tensor q, torch::Tensor k, torch::Tensor v, double scale) {
  TORCH_CHECK(q.dim() == 4);
  auto out = torch::empty({q.size(0), q.size(2), q.size(1) * q.size(3)}, q.options());
  auto lse = torch::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(torch::kFloat32));
  run_prefill(q, k, v, out.view({q.size(0), q.size(2), q.size(1), q.size(3)}).transpose(1, 2), q.size(2), 0, scale, true,
              c10::nullopt, lse.data_ptr<float>());
  return {out, lse};
}
