// Products of a prompt's rows with a bf16 matrix for CDNA4 (gfx950): X [M, K] times W [K, N],
// or W [N, K] transposed (a backward pass), and what follows them: a bias and GELU, a
// residual, or the SwiGLU of a fused gate and up projection.
//
// For tens to some thousands of rows: the library's kernels leave many compute units
// without a tile (758 x 4096 has 48 tiles of 256 x 256) or one with twice the others' work,
// and read weights at 2 TB/s where a prompt of 128 tokens is bound by reading them.
//
// Two kinds of tiles. Those of 160 to 256 rows and 256 columns, of 96 rows, and of 128 x 192, are four waves' (gemm_wide.h), bound by the
// way from L2 to LDS and by the matrix cores. Those for fewer rows or columns, or short K, are eight waves': up to 128 x 256, where one wave's store
// runs beneath another's products (by four waves 2048 x 11264 took 40.8 us at 640 rows, not 37.4, and 1.5% longer over all). BM x BN and K in steps of 64,
// through ST buffers of LDS that are filled straight from memory (buffer_load ... lds: no registers, no stores, and
// what lies beyond the rows or columns repeats the last ones). A step is two phases of 32 of K;
// in each, the matrix cores work on one set of fragments while the next set is read from LDS
// and some of the loads of the step ST - 1 ahead are issued. All loads of a step issued at
// once, behind the barrier, block the waves until the caches' queues have taken them. The barrier leaves the loads of
// later steps in flight. 16-byte groups of LDS rows are permuted by the row, so that the rows that a load
// touches lie in different banks; W [K, N] is read by transposing loads. These are bound by reading weights.
//
// Tiles that fill all compute units are summed over all of K; those left over in the last wave
// of workgroups are split along K, so that it is as full as the others, and a second
// kernel adds their parts up. Each chiplet has its own consecutive run of tiles, rows first: they find
// a run of columns' weights in its L2. The product is W^T X^T, so that a lane ends with 4 neighbouring columns of one row.
//
// MI355X, us, the library's kernels, the best of those of eight waves, and the tile that is chosen, with their sum of
// parts, weights from memory:
//   rows                   128                 512                758               1024
//   4096 x 4096         39, 19, 19          39, 31, 31         41, 40, 40         44, 41, 41
//   4096 x 22016        67, 51, 47          89, 107, 99       134, 134, 128      167, 179, 169
//   11008 x 4096        96, 29, 29          96, 54, 54        101, 86, 69        110, 90, 87
//   16384 x 4096       139, 38, 38         138, 74, 71        146, 120, 92       157, 124, 116
//   28672 x 8192       207, 100, 99        357, 214, 196      307, 376, 295      376, 387, 359
//   22016, transposed, to 4096:  114, 52, 51    234, 102, 89   231, 160, 117      247, 165, 144
//   12288, transposed, to 4096:   66, 32, 32     78, 59, 59     89, 97, 76        109, 99, 91
// A call takes the host 8 us, the library's 18. Which of the two a product takes are ops/prompt_grad.py's rules
// (takes_gemm, takes_wide_gemm); profiles/prompt_products.csv and prompt_products_wide.csv have what they were drawn from.

#include "gemm_wide.h"
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

#define GEMM_BK 64

// byte offset of 16-byte group c in a row of 128 bytes, and of one in a row of W [K, N]
__device__ __forceinline__ int gemm_row_group(int row, int c) { return row * (GEMM_BK * 2) + ((c ^ (row & 7)) << 4); }
template <int BN>
__device__ __forceinline__ int gemm_w_swizzle(int row) {
  constexpr int GROUPS = BN / 8;  // a power of two, at least 16
  return (((row & 3) | ((row >> 1) & 4)) << 1) & (GROUPS - 1);
}

// WT: W is [N, K]. WR x WC waves of 16 FM rows and 16 FN columns.
template <bool WT, int WR, int WC, int FM, int FN, int ST>
__global__ __launch_bounds__(GEMM_THREADS, 2) void gemm_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, GemmShape s, GemmOut o) {
  constexpr int BK = GEMM_BK, BM = WR * FM * 16, BN = WC * FN * 16;
  constexpr int XB = BM * BK * 2, STAGE = XB + BK * BN * 2;
  // loads of 1 KB: of X; of a step; per wave (what is left over repeats the last); in the first phase
  constexpr int XI = XB / 1024, ALL = STAGE / 1024, L = (ALL + 7) / 8, H = (L + 1) / 2;
  static_assert(WR * WC == 8 && ST >= 3);
  extern __shared__ __align__(1024) unsigned char gemm_lds[];

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid & (WAVE - 1);
  const int col = lane & 15, hi = lane >> 4;
  GemmSpot spot;
  if (!gemm_spot(s, s.k / BK, &spot)) return;
  const int tile = spot.tile, first = spot.first, steps = spot.steps, part = spot.part;
  const bool pairs = o.epilogue == GEMM_SWIGLU;
  const GemmPlace place = gemm_place<BN>(s, tile);
  const int m0 = place.row * BM, column_tile = place.column;
  const int wm = wave / WC * FM * 16, wn = wave % WC * FN * 16;

  // this wave's loads: byte offsets of each lane, of the step, and what a step adds
  unsigned lane_at[L], step_at[L], step_size[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int load = min(wave * L + i, ALL - 1);
    if (load < XI) {
      const int p = load * 64 + lane, row = p / 8, c = p % 8 ^ (row & 7);
      lane_at[i] = ((unsigned)min(m0 + row, s.m - 1) * s.k + c * 8) * 2;
      step_size[i] = BK * 2;
    } else if (WT) {
      const int p = (load - XI) * 64 + lane, row = p / 8, c = p % 8 ^ (row & 7);
      const int n = gemm_source_column<FN>(column_tile, row, BN, s.n, pairs);
      lane_at[i] = ((unsigned)min(n, s.n - 1) * s.k + c * 8) * 2;
      step_size[i] = BK * 2;
    } else {
      const int p = (load - XI) * 64 + lane, row = p / (BN / 8), c = p % (BN / 8) ^ gemm_w_swizzle<BN>(row);
      const int n = gemm_source_column<FN>(column_tile, c * 8, BN, s.n, pairs);
      lane_at[i] = ((unsigned)row * s.n + min(n, s.n - 8)) * 2;
      step_size[i] = (unsigned)BK * s.n * 2;
    }
    step_at[i] = first * step_size[i];
  }
  auto resource = [](const void* p, unsigned bytes) {
    const size_t at = (size_t)p;
    return gemm_rsrc{__builtin_amdgcn_readfirstlane((int)at), __builtin_amdgcn_readfirstlane((int)(at >> 32) & 0xFFFF),
                     (int)bytes, 0x00020000};
  };
  const gemm_rsrc xr = resource(x, (unsigned)s.m * s.k * 2), wr = resource(w, (unsigned)s.k * s.n * 2);
  const unsigned base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)gemm_lds;
  auto load = [&](unsigned to, int i) {
    const int n = min(wave * L + i, ALL - 1);
    const gemm_rsrc r = n < XI ? xr : wr;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(to + n * 1024), "v"(lane_at[i]), "s"(r), "s"(step_at[i])
                 : "memory", "m0");
    step_at[i] += step_size[i];
  };

  unsigned xa[2], wa[WT ? 2 : FN];  // addresses of this lane's fragments
#pragma unroll
  for (int kc = 0; kc < 2; ++kc) {
    xa[kc] = base + gemm_row_group(wm + col, kc * 4 + hi);
    if (WT) wa[kc] = base + XB + gemm_row_group(wn + col, kc * 4 + hi);
  }
  if (!WT)
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int row = hi * 8 + col / 4, c = (wn + i * 16) / 8 + ((col >> 1) & 1);
      wa[i] = base + XB + row * (BN * 2) + ((c ^ gemm_w_swizzle<BN>(row)) << 4) + (col & 1) * 8;
    }
  using lds_v4s = __attribute__((address_space(3))) v4s;
  using lds_frag = const __attribute__((address_space(3))) bf16x8;
  f32x4 acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 xf[2][FM] = {}, wf[2][FN] = {};
  auto read = [&](int set, unsigned buf, int n) {  // the n-th fragment, of the step's half `set`
    if (n < FM) {
      xf[set][n] = *(lds_frag*)(size_t)(xa[set] + buf + n * 16 * BK * 2);
    } else if (n < FM + FN) {
      const int i = n - FM;
      if (WT) {
        wf[set][i] = *(lds_frag*)(size_t)(wa[set] + buf + i * 16 * BK * 2);
      } else {
        // rows hi*8 + col/4 and 4 below, which are permuted alike; 4 columns a lane
        const unsigned p = wa[i] + buf + set * 32 * BN * 2;
        const v4s a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(size_t)p);
        const v4s b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(size_t)(p + 4 * BN * 2));
        wf[set][i] = bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      }
    }
  };
  // products of one set; meanwhile the other set is read (half of a step later), and loads
  // [l0, l1) of a later step are issued
  auto phase = [&](bool multiply, int set, bool reads, unsigned buf, bool loads, unsigned to, int l0, int l1) {
    constexpr int EARLY = FN > 1 ? (FM + FN + FN / 2 - 1) / (FN / 2) : FM + FN;  // reads are over half way through
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      if (reads)
#pragma unroll
        for (int e = 0; e < EARLY; ++e) read(set ^ 1, buf, i * EARLY + e);
      if (loads)
#pragma unroll
        for (int l = 0; l < L; ++l)
          if (l >= l0 && l < l1 && (l - l0) * FN / (l1 - l0) == i) load(to, l);
      if (multiply)
#pragma unroll
        for (int j = 0; j < FM; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][i], xf[set][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Step t is whole in LDS, and all waves have read step t - 1, whose buffer is the next to be filled.
  // Loads come back in order: those of the ST - 2 steps after t may be out.
  auto arrive = [&](bool more) {
    if (more)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((ST - 2) * L) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

#pragma unroll
  for (int t = 0; t < ST - 1; ++t)
    if (t < steps)
#pragma unroll
      for (int l = 0; l < L; ++l) load(base + t * STAGE, l);
  unsigned from = 0, to = base + (ST - 1) * STAGE;
  const bool longer = steps >= ST;
  arrive(longer);
  phase(false, 1, true, from, longer, to, 0, H);
  phase(true, 0, true, from, longer, to, H, L);
  int t = 1;
  for (; t + ST - 1 < steps; ++t) {
    from = from + STAGE == ST * STAGE ? 0 : from + STAGE;
    to = to + STAGE == base + ST * STAGE ? base : to + STAGE;
    arrive(true);
    phase(true, 1, true, from, true, to, 0, H);
    phase(true, 0, true, from, true, to, H, L);
  }
  for (; t < steps; ++t) {
    from = from + STAGE == ST * STAGE ? 0 : from + STAGE;
    arrive(false);
    phase(true, 1, true, from, false, to, 0, H);
    phase(true, 0, true, from, false, to, H, L);
  }
  phase(true, 1, false, from, false, to, 0, H);

  if (part >= 0) {
    float* to_part = o.parts + ((size_t)part * s.rest + tile - s.whole) * (BM * BN);
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int i = 0; i < FN; ++i)
        *reinterpret_cast<f32x4*>(to_part + (wm + j * 16 + col) * BN + wn + i * 16 + hi * 4) = acc[i][j];
    return;
  }
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int m = m0 + wm + j * 16 + col;
    if (pairs) {
#pragma unroll
      for (int i = 0; i < FN / 2; ++i)
        gemm_store_pair(s, o, m, gemm_source_column<FN>(column_tile, wn + i * 16 + hi * 4, BN, s.n, true), acc[i][j],
                        acc[i + FN / 2][j]);
    } else {
#pragma unroll
      for (int i = 0; i < FN; ++i) gemm_store(s, o, m, column_tile * BN + wn + i * 16 + hi * 4, acc[i][j]);
    }
  }
}

// ------------------------------------------------------- tiles of four waves

// rows and columns of 16 of a tile. Two rows of waves read less from LDS where rows are many; W [K, N] with few
// rows is 5% faster with one (758 x 4096 x 22016 in tiles of 160 rows: 134.7 us, 143)
template <bool WT, int ROWS, int COLUMNS>
struct WideGemm {
  static constexpr int WR = ROWS % 2 == 0 && (WT || ROWS > 10 || COLUMNS % 8) ? 2 : 1, FM = ROWS / WR, FN = COLUMNS * WR / 4;
  using Tile = WideTile<WT, WR, FM, FN>;
};

template <bool WT, int ROWS, int COLUMNS>
__global__ __launch_bounds__(WIDE_THREADS, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_wide_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, GemmShape s, GemmOut o) {
  using Gemm = WideGemm<WT, ROWS, COLUMNS>;
  using Tile = typename Gemm::Tile;
  constexpr int FM = Gemm::FM, FN = Gemm::FN, BM = Tile::BM, BN = Tile::BN;
  extern __shared__ __align__(1024) unsigned char gemm_lds[];
  GemmSpot spot;
  if (!gemm_spot(s, s.k / GEMM_BK, &spot)) return;
  const bool pairs = o.epilogue == GEMM_SWIGLU;
  const GemmPlace place = gemm_place<BN>(s, spot.tile);
  const int m0 = place.row * BM, column_tile = place.column;
  f32x4 acc[FN][FM];
  wide_product<WT, Gemm::WR, FM, FN>(
      gemm_lds, acc, wide_resource(x, (unsigned)s.m * s.k * 2), wide_resource(w, (unsigned)s.k * s.n * 2),
      [&](int row) { return (unsigned)min(m0 + row, s.m - 1) * s.k * 2; },
      [&](int c) { return (unsigned)min(gemm_source_column<FN>(column_tile, c, BN, s.n, pairs), s.n - (WT ? 1 : 8)); },
      (unsigned)(WT ? s.k : s.n) * 2, spot.first, spot.steps);
  if (spot.part >= 0) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x & (WAVE - 1);
    float* to = o.parts + ((size_t)spot.part * s.rest + spot.tile - s.whole) * (BM * BN) + (wave * FM * FN * WAVE + lane) * 4;
    wide_each<FM>([&](auto j_) {
      constexpr int j = decltype(j_)::value;
      wide_each<FN>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        wide_pin<(j * FN + i < 56)>(acc[i][j]);
        *reinterpret_cast<f32x4*>(to + (j * FN + i) * WAVE * 4) = acc[i][j];
      });
    });
    return;
  }
  // loads of residuals that follow stores wait for a trip to memory each: 16 to 32 of them
  const int row = m0 + wide_row<WT, Gemm::WR, FM, FN>(), c = wide_column<WT, Gemm::WR, FM, FN>();
  int n[FN / 2];
  Gemm8 bias[FN / 2] = {}, residual[2][FN / 2] = {};
#pragma unroll
  for (int i = 0; i < FN / 2; ++i) {
    n[i] = gemm_source_column<FN>(column_tile, c + i * 32, BN, s.n, pairs);
    if (o.bias) bias[i] = gemm_load8(o.bias + min(n[i], s.n - 8));
  }
  wide_store<FM, FN>(
      pairs, acc,
      [&](auto j) {
        if (o.residual)
#pragma unroll
          for (int i = 0; i < FN / 2; ++i)
            residual[j & 1][i] = gemm_load8(o.residual + (size_t)min(row + j * 16, s.m - 1) * s.n + min(n[i], s.n - 8));
      },
      [&](auto j, auto i, float (&v)[8], float (&u)[8]) {
        if (pairs) gemm_store_pair(s, o, row + j * 16, n[i], v, u);
        else gemm_store(s, o, row + j * 16, n[i], v, bias[i], residual[j & 1][i]);
      });
}

// parts [splits, rest, waves, FM, FN, 64, 4]: two fragments, with pairs four, per thread
template <bool WT, int ROWS, int COLUMNS>
__global__ __launch_bounds__(256) void gemm_wide_parts_kernel(GemmShape s, GemmOut o) {
  using Gemm = WideGemm<WT, ROWS, COLUMNS>;
  using Tile = typename Gemm::Tile;
  constexpr int FM = Gemm::FM, FN = Gemm::FN, BM = Tile::BM, BN = Tile::BN;
  const bool pairs = o.epilogue == GEMM_SWIGLU;
  const int unit = __builtin_amdgcn_readfirstlane((blockIdx.x * 256 + threadIdx.x) / WAVE), lane = threadIdx.x & (WAVE - 1);
  const int each = pairs ? FN / 4 : FN / 2, i = unit % each * 2, j = unit / each % FM, wave = unit / each / FM % 4;
  const int tile = unit / each / FM / 4;
  if (tile >= s.rest) return;
  const float* p = o.parts + (size_t)tile * (BM * BN) + (((wave * FM + j) * FN + i) * WAVE + lane) * 4;
  const size_t stride = (size_t)s.rest * (BM * BN);
  f32x4 sum[4] = {};
  for (int k = 0; k < s.splits; ++k)
#pragma unroll
    for (int f = 0; f < 4; ++f)
      if (f < 2 || pairs) sum[f] += *reinterpret_cast<const f32x4*>(p + k * stride + ((f >> 1) * (FN / 2) + (f & 1)) * WAVE * 4);
  const GemmPlace place = gemm_place<BN>(s, s.whole + tile);
  const int hi = lane >> 4, m = place.row * BM + (wave / Tile::WC * FM + j) * 16 + (lane & 15);
  const int n = gemm_source_column<FN>(place.column, (wave % Tile::WC * FN + i + (hi & 1)) * 16 + (hi >> 1) * 8, BN, s.n, pairs);
  float v[8];
  wide_join(sum[0], sum[1], v);
  if (pairs) {
    float u[8];
    wide_join(sum[2], sum[3], u);
    gemm_store_pair(s, o, m, n, v, u);
  } else {
    Gemm8 bias = {}, residual = {};
    if (o.bias) bias = gemm_load8(o.bias + min(n, s.n - 8));
    if (o.residual) residual = gemm_load8(o.residual + (size_t)min(m, s.m - 1) * s.n + min(n, s.n - 8));
    gemm_store(s, o, m, n, v, bias, residual);
  }
}

template <bool WT, int ROWS, int COLUMNS>
static void launch_gemm_wide(const unsigned short* x, const unsigned short* w, const GemmShape& s, const GemmOut& o, long blocks, hipStream_t stream) {
  using Tile = typename WideGemm<WT, ROWS, COLUMNS>::Tile;
  const hipError_t fits = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wide_kernel<WT, ROWS, COLUMNS>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, Tile::LDS);
  TORCH_CHECK(fits == hipSuccess, "gemm_rows: ", hipGetErrorString(fits));
  gemm_wide_kernel<WT, ROWS, COLUMNS><<<blocks, WIDE_THREADS, Tile::LDS, stream>>>(x, w, s, o);
  HIP_CHECK_LAST();
  if (s.splits > 1) {
    const long threads = (long)s.rest * Tile::BM * Tile::BN / (o.epilogue == GEMM_SWIGLU ? 16 : 8);
    gemm_wide_parts_kernel<WT, ROWS, COLUMNS><<<(threads + 255) / 256, 256, 0, stream>>>(s, o);
    HIP_CHECK_LAST();
  }
}

// ------------------------------------------------------------------- host

// step, fixed and alone by least squares over 1539 products of the presets, 17 to 4096 rows, in either direction, with what
// follows: 7% off in the mean. The tile that they choose takes 1.0% more than the best one, 1.4% for matrices of up to 25 million
// weights (profiles/prompt_products_wide.csv)
static const GemmTile GEMM_TILES[] = {{128, 256, 0.863f, 6.7f, 0.82f}, {128, 128, 0.554f, 4.6f, 0.96f}, {64, 256, 0.668f, 5.9f, 1.f},
                                      {32, 256, 0.564f, 4.4f, 1.f},    {256, 256, 1.469f, 5.f, 0.84f},  {192, 256, 1.205f, 5.3f, 0.75f},
                                      {160, 256, 1.032f, 6.f, 0.7f},   {96, 256, 0.782f, 5.5f, 0.92f},  {128, 192, 0.73f, 5.3f, 0.9f}};

// For what a router reads: the first four tiles alone, by the cost of their steps alone. A sum that is cut along K elsewhere is as
// exact but rounds otherwise now and then, which sends a token to the other of two experts that score alike. So these products keep
// their cuts whatever is measured for the others, and whoever has a router asks for it (`steady`).
static const GemmTile GEMM_STEADY[] = {{128, 256, 0.92f}, {128, 128, 0.55f}, {64, 256, 0.65f}, {32, 256, 0.5f}};

// x [M, K] bf16, w [K, N] (or [N, K], transposed) bf16 -> [M, N] bf16 (swiglu: [M, N/2])
torch::Tensor gemm_rows(torch::Tensor x, torch::Tensor w, bool transposed, int64_t epilogue,
                        c10::optional<torch::Tensor> residual, c10::optional<torch::Tensor> bias, int64_t tile, bool steady) {
  for (const auto& t : {x, w})
    TORCH_CHECK(t.is_cuda() && t.dtype() == torch::kBFloat16 && t.dim() == 2 && t.is_contiguous() &&
                reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "gemm_rows takes aligned bf16 matrices");
  TORCH_CHECK(w.device() == x.device());
  const long m = x.size(0), k = x.size(1), n = w.size(transposed ? 0 : 1);
  TORCH_CHECK(w.size(transposed ? 1 : 0) == k, "gemm_rows: shapes differ");
  const bool pairs = epilogue == GEMM_SWIGLU;
  TORCH_CHECK(epilogue >= 0 && epilogue <= 3 && k >= GEMM_BK && k % GEMM_BK == 0 && n >= 8 && n % (pairs ? 16 : 8) == 0,
              "gemm_rows: sizes out of range");
  // offsets into either are 32-bit
  TORCH_CHECK(m * k < (1L << 31) && k * n < (1L << 31) && m < (1L << 24), "gemm_rows: too large");
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
  steady = steady && tile < 0;
  const GemmTile* const tiles = steady ? GEMM_STEADY : GEMM_TILES;
  const int count = steady ? sizeof(GEMM_STEADY) / sizeof(GemmTile) : sizeof(GEMM_TILES) / sizeof(GemmTile);
  for (int i = 0; i < count; ++i) {
    if (tile >= 0 ? tile != i : pairs && tiles[i].bn == 192) continue;
    float us;
    const GemmShape p = gemm_plan(m, n, k, GEMM_BK, 8, tiles[i], &us);
    if (s.m == 0 || us < least) best = i, least = us, s = p;
  }
  const GemmTile& t = tiles[best];
  TORCH_CHECK(s.m && !(pairs && t.bn == 192), "gemm_rows: no such tile");  // 96 gates would not be whole pairs of fragments
  torch::Tensor parts;
  if (s.splits > 1) {
    parts = torch::empty({(long)s.splits * s.rest * t.bm * t.bn}, x.options().dtype(torch::kFloat32));
    o.parts = parts.data_ptr<float>();
  }
  const long blocks = s.whole + ((long)s.rest * s.splits + 7) / 8 * 8;
  TORCH_CHECK(blocks < (1L << 31));
  auto stream = at::cuda::getCurrentCUDAStream();
#define GEMM(WT, WR, WC, FM, FN, ST)                                                                                \
  do {                                                                                                              \
    constexpr int BM = WR * FM * 16, BN = WC * FN * 16, LDS = ST * (BM + BN) * GEMM_BK * 2;                         \
    TORCH_CHECK(BM == t.bm && BN == t.bn);                                                                          \
    const hipError_t fits = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_kernel<WT, WR, WC, FM, FN, ST>), \
                                                hipFuncAttributeMaxDynamicSharedMemorySize, LDS);                   \
    TORCH_CHECK(fits == hipSuccess, "gemm_rows: ", hipGetErrorString(fits));                                        \
    gemm_kernel<WT, WR, WC, FM, FN, ST><<<blocks, GEMM_THREADS, LDS, stream>>>(BF16P(x), BF16P(w), s, o);           \
    HIP_CHECK_LAST();                                                                                               \
    if (s.splits > 1) {                                                                                             \
      const long threads = (long)s.rest * BM * (pairs ? BN / 2 : BN) / 4;                                           \
      gemm_parts_kernel<BM, BN, FN><<<(threads + 255) / 256, 256, 0, stream>>>(s, o);                               \
      HIP_CHECK_LAST();                                                                                             \
    }                                                                                                               \
  } while (0)
#define GEMM_EITHER(...)                       \
  do {                                         \
    if (transposed) GEMM(true, __VA_ARGS__);   \
    else GEMM(false, __VA_ARGS__);             \
  } while (0)
#define GEMM_WIDE(ROWS, COLUMNS)                                                                             \
  do {                                                                                              \
    TORCH_CHECK(ROWS * 16 == t.bm && COLUMNS * 16 == t.bn);                                                          \
    if (transposed) launch_gemm_wide<true, ROWS, COLUMNS>(BF16P(x), BF16P(w), s, o, blocks, stream);         \
    else launch_gemm_wide<false, ROWS, COLUMNS>(BF16P(x), BF16P(w), s, o, blocks, stream);                   \
  } while (0)
  switch (best) {
    case 0: GEMM_EITHER(2, 4, 4, 4, 3); break;
    case 1: GEMM_EITHER(2, 4, 4, 2, 4); break;
    case 2: GEMM_EITHER(2, 4, 2, 4, 4); break;
    case 3: GEMM_EITHER(1, 8, 2, 2, 4); break;
    case 4: GEMM_WIDE(16, 16); break;
    case 5: GEMM_WIDE(12, 16); break;
    case 6: GEMM_WIDE(10, 16); break;
    case 7: GEMM_WIDE(6, 16); break;
    case 8: GEMM_WIDE(8, 12); break;
  }
#undef GEMM_WIDE
#undef GEMM_EITHER
#undef GEMM
  return y;
}
