// Products of a prompt's rows with NF4 weights for CDNA4 (gfx950): X [M, K] in bf16 times tiles of codes
// (nf4_tiles.hip has their order), and what follows them, as in gemm.hip. A weight is level * scale, rounded to
// bf16, as a copy of the matrix in bf16 would hold it: no such copy is made, kept or read, which is what bounds
// products of up to 128 rows by gemm.hip (4.9 TB/s; where there is no copy, its making comes first, 33 us for 8192 x 8192, 230 for 8192 x 57344).
//
// A workgroup of 8 waves has 32 FM rows and 256 columns, 32 of each wave, whose weights that wave makes in its
// registers, where they are the matrix cores' operand: of 16 bytes of codes a lane has two runs of 8 inputs of
// one column. Both levels of a byte come from a table in LDS, which is there 32 times, so that the
// lanes of half a wave read from banks of their own (5.3 cycles a look-up; 6.6 from one table). Rows come through
// registers to two tiles in LDS, scales to LDS as 32-bit numbers (converted where they are used, 64 more vector
// operations a tile: 5 to 10% slower).
//
// Matrix instructions of 32 x 32, as vector instructions run beside these (6 in 32 cycles at no cost) and hardly
// beside those of 16 x 16 (3 in 16 cycles cost what they cost alone: 128 x 8192 x 57344 took 174 us with them, 139 now, 150 among a prompt's other launches).
// A step is 16 inputs: its products, among which the next step's weights are rounded, those of the third
// after it looked up, and rows read. Up to 32 rows it is bound by LDS (look-ups and scales: 2000 of 2600 cycles a tile of
// 128 inputs), with 128 by the matrix cores with vector instructions beside them (0.86 PFLOP/s, 1.0 in the workgroups
// that there are: 224 on 256 compute units). Four waves of 64 columns, with half as many reads of rows and one wave on a
// SIMD: 236 us.
//
// MI355X, us, gemm.hip or the library with copies that are there already, and this one with its sum of parts:
//   rows                    16            64           128          192
//   8192 x 10240        37.8, 24.9    39.8, 31.5   44.9, 42.8   62.9, 54.9
//   8192 x 57344 gated   168, 78       170, 96      178, 150     204, 282
//   28672 x 8192        85.2, 44.8    89.2, 54.7   96.6, 79.4    131, 136
//   4096 x 6144         17.1, 16.4    19.9, 21.7   21.9, 26.5   28.6, 29.6

#include "gemm.h"
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

#define NF4_BK 128       // inputs of a tile of codes
#define NF4_BN 256       // columns of a workgroup: 8 waves of two runs of 16
#define NF4_COPIES 32    // of the table

static __device__ __constant__ float NF4_GEMM_LEVELS[16] = {
    -1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f,
    -0.28444138169288635f, -0.18477343022823334f, -0.09105003625154495f, 0.0f,
    0.07958029955625534f, 0.16093020141124725f, 0.24611230194568634f,
    0.33791524171829224f, 0.4407098293304443f, 0.5626170039176941f,
    0.7229568362236023f, 1.0f};

// byte offset of 16-byte group c in a row of 256 bytes
__device__ __forceinline__ int nf4_row_group(int row, int c) { return row * (NF4_BK * 2) + ((c ^ (row & 15)) << 4); }

// FM x 32 rows and 256 columns, 32 of each wave; D tiles of codes and of X ahead. PAIRS: half of a wave's columns are
// gates, half ups
template <int FM, int D, bool PAIRS>
__global__ __launch_bounds__(512, 2) void nf4_gemm_kernel(
    const unsigned short* __restrict__ x, const uint4* __restrict__ tiles, const unsigned short* __restrict__ scales,
    GemmShape s, GemmOut o) {
  constexpr int BM = FM * 32, BN = NF4_BN, NS = PAIRS ? 2 : 1;
  constexpr int TABLE = 256 * NF4_COPIES * 8, XB = BM * NF4_BK * 2, XN = FM;
  constexpr int XD = FM == 4 ? 1 : 2, XS = 2 * XD;  // steps that rows are read and codes looked up ahead
  constexpr int SB = NF4_BK * 4;  // of scales, in 32 bits
  // table, two tiles of X, two of scales of each wave. Not extern: at an address that the compiler knows, which saves an
  // addition for each look-up
  __shared__ __align__(1024) unsigned char lds[TABLE + 2 * XB + 8 * 2 * NS * SB];

  GemmSpot spot;
  if (!gemm_spot(s, s.k / NF4_BK, &spot)) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid & (WAVE - 1);
  const int col = lane & 31, hi = lane >> 5;
  const GemmPlace place = gemm_place<NF4_BN>(s, spot.tile);
  const int m0 = place.row * BM, column_tile = place.column;
  const int n_kb = s.k / NF4_BK, last = spot.first + spot.steps - 1;

  // of a tile of codes, this lane has 2 of the 4 runs of 16 inputs (in either half of the tile) of one column
  const int n = gemm_source_column<2>(column_tile, wave * 32 + (col & 16), BN, s.n, PAIRS);
  const int run = min(n, s.n - 16) / 16;
  const uint4* wp = tiles + ((size_t)(run / 4) * n_kb * 4 + run % 4) * 64 + hi * 32 + (lane & 15);
  const unsigned short* sp = scales + (size_t)(run / 4) * n_kb * NF4_BK + (lane & 15) * 8;
  const unsigned short* xp[XN];
  int xat[XN];
#pragma unroll
  for (int i = 0; i < XN; ++i) {
    const int row = (tid + i * 512) / 16, c = tid % 16;
    xp[i] = x + (size_t)min(m0 + row, s.m - 1) * s.k + c * 8;
    xat[i] = TABLE + nf4_row_group(row, c);
  }
  const int scale_to = TABLE + 2 * XB + wave * (2 * NS * SB), lane8 = col * 8;
  const int scale_at = scale_to + (PAIRS ? col / 16 * SB : 0) + hi * 128;
  u32x4 codes[D][2], scale[D];
  bf16x8 xs[D][XN];
  auto fetch_x = [&](int kb, int d) {
    const int at = min(kb, last) * NF4_BK;
#pragma unroll
    for (int i = 0; i < XN; ++i) xs[d][i] = *reinterpret_cast<const bf16x8*>(xp[i] + at);
  };
  auto fetch_w = [&](int kb, int d) {
    const int at = min(kb, last);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      codes[d][i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp + (size_t)at * 256 + i * 16));
    scale[d] = *reinterpret_cast<const u32x4*>(sp + at * NF4_BK);
  };
  auto stage_x = [&](int buf, int d) {
#pragma unroll
    for (int i = 0; i < XN; ++i) *reinterpret_cast<bf16x8*>(lds + xat[i] + buf * XB) = xs[d][i];
  };
  auto stage_scale = [&](int buf, int d) {  // lanes 0 to 15: those of gates or of all, 16 to 31: of ups
    if (lane < 16 * NS) {
      f32x4* to = reinterpret_cast<f32x4*>(lds + scale_to + buf * (NS * SB) + lane * 32);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const unsigned a = scale[d][2 * i], b = scale[d][2 * i + 1];
        to[i] = f32x4{__uint_as_float(a << 16), __uint_as_float(a & 0xFFFF0000u), __uint_as_float(b << 16), __uint_as_float(b & 0xFFFF0000u)};
      }
    }
  };

  using f32x16 = __attribute__((ext_vector_type(16))) float;
  f32x16 acc[FM];
#pragma unroll
  for (int j = 0; j < FM; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
  bf16x8 xf[XS][FM], wf[2];
  float2 level[2][4];
  f32x4 sc[2][2];
  // step t of a tile, 16 inputs: a lane has 8 of them, group t%4/2*8 + (hi*2 + t/4)*2 + t%2 of 16
  auto read_x = [&](int buf, int t, int j) {
    xf[t & (XS - 1)][j] = *reinterpret_cast<const bf16x8*>(
        lds + TABLE + buf * XB + nf4_row_group(j * 32 + col, t % 4 / 2 * 8 + (hi * 2 + t / 4) * 2 + t % 2));
  };
  auto read_scales = [&](int buf, int t) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      sc[t & 1][i] = *reinterpret_cast<const f32x4*>(lds + scale_at + buf * (NS * SB) + (t % 4 / 2 * 8 + t / 4 * 2 + t % 2) * 32 + i * 16);
  };
  auto look_up = [&](int d, int t) {
    const unsigned w = codes[d][t / 4][t % 4];
#pragma unroll
    for (int b = 0; b < 4; ++b)  // byte b times 256, and this lane's copy
      level[t & 1][b] = *reinterpret_cast<const float2*>(lds + __builtin_amdgcn_perm(w, lane8, 0x0C0C0400u + (b << 8)));
  };
  auto round = [&](int t) {  // what was looked up, as weights
    using f32x8 = __attribute__((ext_vector_type(8))) float;
    using bf8 = __attribute__((ext_vector_type(8))) __bf16;
    f32x8 v;
#pragma unroll
    for (int b = 0; b < 8; ++b) v[b] = (b < 4 ? level[t & 1][b & 3].x : level[t & 1][b & 3].y) * sc[t & 1][b / 4][b % 4];
    wf[t & 1] = __builtin_bit_cast(bf16x8, __builtin_convertvector(v, bf8));
  };

#pragma unroll
  for (int d = 0; d < D; ++d) {
    fetch_x(spot.first + d, d);
    fetch_w(spot.first + d, d);
  }
  // both levels of a byte, once for each of 32 lanes: these read from as many banks
  const float low = NF4_GEMM_LEVELS[tid / NF4_COPIES];
#pragma unroll
  for (int i = 0; i < 16; ++i) *reinterpret_cast<float2*>(lds + (i * 512 + tid) * 8) = make_float2(low, NF4_GEMM_LEVELS[i]);
  stage_x(0, 0);
  stage_scale(0, 0);
  fetch_x(spot.first + D, 0);
  __syncthreads();
  read_scales(0, 0);
  look_up(0, 0);
  round(0);
#pragma unroll
  for (int t = 1; t <= 2; ++t) {
    look_up(0, t);
    read_scales(0, t);
  }
#pragma unroll
  for (int t = 0; t < XD; ++t)
#pragma unroll
    for (int j = 0; j < FM; ++j) read_x(0, t, j);
  // Products of a step; among them the next one's weights are rounded, those of the third after it looked up,
  // and rows of later ones read. The next tile's rows are written in step 2, seen once they are read.
  for (int kb = spot.first; kb <= last; kb += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {  // tile kb + d
      if (d && kb + d > last) break;
      const int next = (d + 1) % D, buf = d & 1;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        if (t == 2) {
          stage_x(buf ^ 1, next);
          stage_scale(buf ^ 1, next);
          fetch_x(kb + d + 1 + D, next);
        }
        if (t == 5) fetch_w(kb + d + D, d);
        if (t == 8 - XD) __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        round(t + 1);
        look_up(t < 5 ? d : next, (t + 3) & 7);
        read_scales(t < 5 ? buf : buf ^ 1, (t + 3) & 7);
#pragma unroll
        for (int j = 0; j < FM; ++j) read_x(t + XD < 8 ? buf : buf ^ 1, (t + XD) & 7, j);
#pragma unroll
        for (int j = 0; j < FM; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[t & 1], xf[t & (XS - 1)][j], acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, (20 + FM - 1) / FM, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, (6 + FM + FM - 1) / FM, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // a lane has columns 8 g + 4 hi + 0..3 of one row
  const int wn = wave * 32 + hi * 4;
  auto four = [&](int j, int g) { return f32x4{acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]}; };
  if (spot.part >= 0) {
    float* to_part = o.parts + ((size_t)spot.part * s.rest + spot.tile - s.whole) * (BM * BN);
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(to_part + (j * 32 + col) * BN + wn + g * 8) = four(j, g);
    return;
  }
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int m = m0 + j * 32 + col;
    if (PAIRS) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
        gemm_store_pair(s, o, m, gemm_source_column<2>(column_tile, wn + g * 8, BN, s.n, true), four(j, g), four(j, g + 2));
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) gemm_store(s, o, m, column_tile * BN + wn + g * 8, four(j, g));
    }
  }
}

// ------------------------------------------------------------------- host

static const GemmTile NF4_GEMM_TILES[] = {{128, NF4_BN, 2.05f}, {64, NF4_BN, 1.37f}, {32, NF4_BN, 1.07f}};

// x [M, K] bf16, tiles and scales of [K, N] -> [M, N] bf16 (swiglu: [M, N/2])
torch::Tensor gemm_nf4_rows(torch::Tensor x, torch::Tensor tiles, torch::Tensor scales, int64_t epilogue,
                            c10::optional<torch::Tensor> residual, c10::optional<torch::Tensor> bias, int64_t tile) {
  TORCH_CHECK(x.is_cuda() && x.dtype() == torch::kBFloat16 && x.dim() == 2 && x.is_contiguous() &&
              reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0, "gemm_nf4_rows takes aligned bf16 rows");
  TORCH_CHECK(tiles.is_cuda() && tiles.dtype() == torch::kUInt8 && tiles.dim() == 5 && tiles.is_contiguous() &&
              tiles.size(2) == 4 && tiles.size(3) == 64 && tiles.size(4) == 16 &&
              reinterpret_cast<uintptr_t>(tiles.data_ptr()) % 16 == 0, "gemm_nf4_rows takes NF4 tiles");
  const long m = x.size(0), k = x.size(1), n = tiles.size(0) * 64;
  TORCH_CHECK(scales.is_cuda() && scales.dtype() == torch::kBFloat16 && scales.dim() == 2 && scales.is_contiguous() &&
              scales.size(0) == tiles.size(0) && scales.size(1) == tiles.size(1) * NF4_BK &&
              reinterpret_cast<uintptr_t>(scales.data_ptr()) % 16 == 0, "scales are those of the tiles");
  TORCH_CHECK(tiles.device() == x.device() && scales.device() == x.device());
  TORCH_CHECK(k >= NF4_BK && k % NF4_BK == 0 && k == tiles.size(1) * NF4_BK, "gemm_nf4_rows: rows are not the tiles'");
  const bool pairs = epilogue == GEMM_SWIGLU;
  TORCH_CHECK(epilogue >= 0 && epilogue <= 3 && n >= 64 && k * n < (1L << 37) && n < (1L << 30) && m < (1L << 24),
              "gemm_nf4_rows: sizes out of range");
  TORCH_CHECK((epilogue == GEMM_RESIDUAL) == residual.has_value(), "a residual belongs to its epilogue");
  auto y = torch::empty({m, pairs ? n / 2 : n}, x.options());
  if (m == 0) return y;
  GemmOut o{BF16P(y), nullptr, nullptr, nullptr, (int)epilogue};
  if (residual.has_value()) {
    TORCH_CHECK(residual->is_cuda() && residual->dtype() == torch::kBFloat16 && residual->is_contiguous() &&
                residual->numel() == m * n && reinterpret_cast<uintptr_t>(residual->data_ptr()) % 8 == 0);
    o.residual = BF16P(*residual);
  }
  if (bias.has_value()) {
    TORCH_CHECK(!pairs && epilogue != GEMM_PLAIN && bias->is_cuda() && bias->dtype() == torch::kBFloat16 && bias->is_contiguous() &&
                bias->numel() == n && reinterpret_cast<uintptr_t>(bias->data_ptr()) % 8 == 0);
    o.bias = BF16P(*bias);
  }
  int best = 0;
  float least = 0.f;
  GemmShape s{};
  for (int i = 0; i < 3; ++i) {
    if (tile >= 0 && tile != i) continue;
    float us;
    const GemmShape p = gemm_plan(m, n, k, NF4_BK, 4, NF4_GEMM_TILES[i], &us);
    if (s.m == 0 || us < least) best = i, least = us, s = p;
  }
  torch::Tensor parts;
  if (s.splits > 1) {
    parts = torch::empty({(long)s.splits * s.rest * NF4_GEMM_TILES[best].bm * NF4_BN}, x.options().dtype(torch::kFloat32));
    o.parts = parts.data_ptr<float>();
  }
  const long blocks = s.whole + ((long)s.rest * s.splits + 7) / 8 * 8;
  TORCH_CHECK(blocks < (1L << 31));
  auto stream = at::cuda::getCurrentCUDAStream();
#define NF4_GEMM(FM, D, PAIRS)                                                                                       \
  do {                                                                                                             \
    constexpr int BM = FM * 32, BN = NF4_BN;                                                                       \
    TORCH_CHECK(BM == NF4_GEMM_TILES[best].bm);                                                                    \
    nf4_gemm_kernel<FM, D, PAIRS><<<blocks, 512, 0, stream>>>(                                                   \
        BF16P(x), reinterpret_cast<const uint4*>(tiles.data_ptr()), BF16P(scales), s, o);                          \
    HIP_CHECK_LAST();                                                                                              \
    if (s.splits > 1) {                                                                                            \
      const long threads = (long)s.rest * BM * (PAIRS ? BN / 2 : BN) / 4;                                          \
      gemm_parts_kernel<BM, BN, 2><<<(threads + 255) / 256, 256, 0, stream>>>(s, o);                               \
      HIP_CHECK_LAST();                                                                                            \
    }                                                                                                              \
  } while (0)
#define NF4_GEMM_EITHER(...)                     \
  do {                                           \
    if (pairs) NF4_GEMM(__VA_ARGS__, true);      \
    else NF4_GEMM(__VA_ARGS__, false);           \
  } while (0)
  switch (best) {
    case 0: NF4_GEMM_EITHER(4, 2); break;
    case 1: NF4_GEMM_EITHER(2, 4); break;
    case 2: NF4_GEMM_EITHER(1, 4); break;
  }
#undef NF4_GEMM_EITHER
#undef NF4_GEMM
  return y;
}
