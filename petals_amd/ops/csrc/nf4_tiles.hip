// Products of few rows with NF4 weights on the matrix cores, in whole numbers.
//
// A 4-bit level times 7783094 is a whole number up to 9.4e-8 of itself (no other factor below
// 127.4 * 2^16 fits all 16 levels as well; a 32-bit product of level, scale and input is
// rounded twice by up to 6e-8), and a whole number is three signed digits of base 256. So is
// an input times its block's scale, rounded to four digits, once the inputs of a run are
// scaled by one power of two so that their largest reaches 2^29. Inputs beyond 64 times the
// run's mean size would leave the others few places; those runs leave out what is too large
// and multiply it in 32-bit floats, one by one (see `strip`), so that a last place is at most
// 2^-22 of a mean that they have no part in. Sums of products of digits are exact
// in 32 bits for runs of 512, and a product of 16 columns with 64 inputs is one
// v_mfma_i32_16x16x64_i8 per digit of the levels: the four digits of up to four rows are its
// other 16 columns. Those of up to eight rows are the other columns of a v_mfma_i32_32x32x32_i8.
//
// Digits come from v_perm_b32, which looks four codes up in eight bytes at once. Two
// lookups make up the 16 levels: a code of the other half selects a sign or a constant (0
// for 12, all ones above), which for given tables is known, and which the other table is
// xored with below, so that the xor of both lookups is the digit; or the tables are made for
// their sum, and both are multiplied (see SUMMED). That costs the same for
// one row as for four, and no LDS, where the kernel that it stands for gathers the two
// levels of a byte from a table: there random indices collide, and every row more is
// another operation a weight.
//
//   tiles   [out/64, ceil(in/128), 4, 64 lanes, 16 bytes]: 128 inputs x 64 columns, in the
//           order of the operands: lane l of part c has column c*16 + l%16, and of each 64
//           inputs the 16 from (l/16)*16 on: bytes 0-3 of a half have the first four in
//           their low and the next four in their high nibbles, bytes 4-7 the rest
//   scales  [out/64, ceil(in/128)*128] bf16, zero beyond `in`
//
// Four waves of a workgroup take 64 columns and 512 inputs each (256 at a time beyond four
// rows, whose digits fill twice the columns), all of whose weights are on their way while
// the inputs are cut into digits. Five to eight rows stay for up to 1024 inputs, as long
// as that leaves 2048 waves: their sums are 96 registers to combine at the end.
//
// Loads have no conditions: what is not there lies beyond the end of a buffer, which gives zeros. With
// conditions a wave's loads were some dozens of branches, each with its own (8192 x 8192, 1 row: 14.9 us, 10.4 now). Digits of
// one input are written together and made columns by loads that transpose bytes; transposed in registers they
// were 8 lookups' worth of instructions for 4 inputs, and stores of 4 bytes whose lanes met in the same banks.
//
// It is bound by vector instructions, not by memory: of 34 for 16 weights of a lane 24 are lookups. A matrix
// instruction keeps others from starting for some 9 cycles, whatever its size; they are spread among the lookups
// (1024 weights took 238 cycles with three waves on a SIMD as the compiler orders them, 197 so; 216 with
// both lookups xored and half as many). llama-2-70b, us a product without its reduction, before this and now, for
// 1, 4 and 8 rows:
//   qkv   8192 x 10240   18.8, 19.7, 27.4     14.6, 15.9, 23.3
//   o     8192 x 8192    14.9, 16.4, 18.9     10.5, 11.9, 16.4
//   gate  8192 x 57344   58.8, 69.3, 96.2     51.3, 62.9, 87.7
//   down  28672 x 8192   31.8, 38.6, 56.6     27.2, 33.7, 50.9
// Workgroups that stay for several runs of columns, with the next one's weights on their way, keep two waves on a
// SIMD: 62 us for the third, 1 row, and as long as now with eight. Four waves a SIMD: 71 beside 65 us then.
// Cut off instead of rounded, and with the largest input of a run at 2^30 whatever the others
// are, it took 0 to 5% less (8192 x 8192: 14.7, 16.1, 18.5 us without the reduction for 1, 4,
// 8 rows beside 14.8, 16.6, 19.5). Runs with inputs beyond 64 times their mean take longer: two
// of 8192 inputs a thousand times the rest, 15.2, 18.2, 23.6.
// Weights are read once and marked so (non-temporal): 2% of a decoding step of four blocks of width
// 8192 with one row (601 to 589 us when it was measured), 1% with eight, 3.5% of two blocks of 8 experts.
// Error against 64 bits, of the root mean square result: 0.9e-7 (nf4.hip: 1.6e-7).

#include "common.h"
#include "gemv_reduce.h"
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>

using i32x4 = __attribute__((ext_vector_type(4))) int;
using u32x4 = __attribute__((ext_vector_type(4))) unsigned;
using i32x2 = __attribute__((ext_vector_type(2))) int;

#define NF4_UNIT (1.0f / 7783094.0f)
// times a run's mean size. Channels ten times as loud as the rest stay below it; with 16 they
// didn't, and 8 rows of 8192 x 57344 took 197 us (the loud ones then in loops of their own)
#define NF4_GATE 64.f
#define NF4_ONCE 2           // of a load: non-temporal
#define NF4_BEYOND (1 << 30)  // bytes, more than a launch has of a run of columns
#define NF4_LAUNCH (1 << 17)  // tiles of 128 inputs, a multiple of a workgroup's, that offsets of 32 bits hold with room for the former
#define NF4_FINITE 0x7F7FFFFFu  // bits of the largest number

static __device__ __constant__ float NF4_TILE_LEVELS[16] = {
    -1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f,
    -0.28444138169288635f, -0.18477343022823334f, -0.09105003625154495f, 0.0f,
    0.07958029955625534f, 0.16093020141124725f, 0.24611230194568634f,
    0.33791524171829224f, 0.4407098293304443f, 0.5626170039176941f,
    0.7229568362236023f, 1.0f};

// digits of the levels, lowest first: bytes 0-3 and 4-7 of the tables of codes 0-7 and 8-15,
// each xored with what the other one yields for a code that is not its own
__device__ constexpr unsigned NF4_DIGITS[3][4] = {
    {0x70a4dab5u, 0xff2a9c36u, 0x7584b78au, 0x4926eac6u},
    {0x19a4ad3du, 0xffcff138u, 0xddc51d8cu, 0x3c232e57u},
    {0x2e3d5289u, 0xff0a15deu, 0xd71d1309u, 0x88a9bc34u},
};
// the same digits as sums of both lookups: less what the other one yields
__device__ constexpr unsigned NF4_SUMMANDS[3][4] = {
    {0x715bdb4bu, 0x01d66436u, 0x8a7bb776u, 0xb7da16c6u},
    {0x1aa5523du, 0x01310f38u, 0x223a1d73u, 0xc4ddd257u},
    {0xd1c2ad89u, 0x01f6ebdeu, 0x281e140au, 0x78574434u},
};

__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// sum, or largest of numbers from zero on, over a wave, the same for all lanes. Bits, as the
// compiler takes what comes out of float arithmetic for finite.
template <bool MAX>
__device__ __forceinline__ unsigned wave_all(float v) {
#define STEP(ctrl, rows)                                                                                   \
  do {                                                                                                     \
    const float other = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, rows, 0xf, false)); \
    v = MAX ? fmaxf(v, other) : v + other;                                                                 \
  } while (0)
  STEP(0xB1, 0xf);   // quads: neighbours
  STEP(0x4E, 0xf);   // quads: pairs
  STEP(0x141, 0xf);  // halves of a row mirrored
  STEP(0x140, 0xf);  // rows of 16 mirrored
  STEP(0x142, 0xa);  // row 0 to 1, 2 to 3
  STEP(0x143, 0xc);  // rows 0 and 1 to 2 and 3
#undef STEP
  return (unsigned)__builtin_amdgcn_readlane(__float_as_int(v), 63);
}

__device__ __forceinline__ float quad_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));
}

// B rows; a wave takes KB tiles of 128 inputs and 64 columns at a time, `steps` times if LONG.
// Grid: (out/64, runs of 4 KB `steps` tiles, rows of sel). With sel, B is 1 and row
// blockIdx.z is that of x[blockIdx.z / k_per_tok] and expert sel[blockIdx.z]. A launch has in_dim inputs
// of x_stride, and n_kb tiles of kb_stride.
template <int B, int KB>
__global__ __launch_bounds__(256, B <= 4 ? 3 : 2) void gemv_nf4_tiles_kernel(
    const uint4* __restrict__ tiles, const unsigned short* __restrict__ scales,
    const float* __restrict__ x,      // [rows, in]
    const int* __restrict__ sel,      // [rows * k_per_tok] or null
    float* __restrict__ partials,     // [splits, B or gridDim.z, out]
    int in_dim, int out_dim, int n_kb, int n_steps, int k_per_tok, int experts, bool by4, int x_stride, int kb_stride) {
  constexpr bool LONG = B > 4;
  const int steps = LONG ? n_steps : 1;
  constexpr bool WIDE = B > 4;  // 32 columns of digits
  constexpr int PER = KB * 2;
  // the two lookups of a digit are multiplied one by one, which saves their xor, where the matrix cores
  // have little else to do
  constexpr bool SUMMED = !WIDE;
  static_assert(KB == (WIDE ? 2 : 4));  // a lane's inputs are 8 slots of 16 bytes
  __shared__ __align__(16) unsigned char digits[4][64 * 128];
  __shared__ __align__(16) float red[4 * B * 64];  // [waves, rows, columns]

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid & (WAVE - 1);
  const int col = lane & 15, hi = lane >> 4;
  const int nb = blockIdx.x, kb0 = (blockIdx.y * 4 + wave) * KB * steps;
  if (sel) {
    const int e = sel[blockIdx.z];
    if (e < 0 || e >= experts) return;  // uniform over the workgroup
    tiles += (size_t)e * (out_dim / 64) * kb_stride * 256;
    scales += (size_t)e * (out_dim / 64) * kb_stride * 128;
    x += (size_t)(blockIdx.z / k_per_tok) * x_stride;
  }

  // loads of what lies beyond a run of columns' inputs, and all of a step that is not there, give zeros
  auto resource = [&](const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
  };
  // inputs of a step: PER of this lane
  auto fetch_x = [&](int step, int b, float* v, int beyond = 0) {
    const auto r = resource(x + (size_t)b * x_stride, (size_t)in_dim * 4);
    const int at = ((kb0 + step * KB) * 128 + lane * PER) * 4 + beyond;
    if (by4) {
#pragma unroll
      for (int i = 0; i < PER; i += 4)
        *reinterpret_cast<u32x4*>(v + i) = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at + i * 4, 0, 0));
    } else {
#pragma unroll
      for (int i = 0; i < PER; ++i) v[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, at + i * 4, 0, 0));
    }
  };
  const auto scale_rsrc = resource(scales + (size_t)nb * kb_stride * 128, (size_t)n_kb * 256);
  auto fetch_scales = [&](int step, unsigned* v, int beyond = 0) {
    const int at = ((kb0 + step * KB) * 128 + lane * PER) * 2 + beyond;
    if constexpr (PER == 8) {
      *reinterpret_cast<u32x4*>(v) = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(scale_rsrc, at, 0, 0));
    } else {
      static_assert(PER == 4);
      using u32x2 = __attribute__((ext_vector_type(2))) unsigned;
      *reinterpret_cast<u32x2*>(v) = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(scale_rsrc, at, 0, 0));
    }
  };
  // operands of 64 inputs and 16 columns, or of 32 inputs, in two runs of 16, and 32 columns
  const auto w_rsrc = resource(tiles + (size_t)nb * kb_stride * 256, (size_t)n_kb * 4096);
  const int w_at = kb0 * 4096 + (WIDE ? (hi & 1) * 64 + (hi >> 1) * 32 + col : lane) * 16;
  u32x4 w[KB][4];
  auto fetch_w = [&](int step, int j, int beyond = 0) {
    const int at = w_at + (step * KB + j) * 4096 + beyond;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      w[j][c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              w_rsrc, at + (WIDE ? c / 2 * 2048 + c % 2 * 256 : c * 1024), 0, NF4_ONCE));
  };

  // all inputs, then the first step's weights, which are awaited last
  constexpr int STEPS = LONG ? 4 : 1;
  float later[STEPS][B][PER];  // of steps 1 on
  unsigned later_scales[STEPS][PER / 2];
  float xs[B][PER];
  unsigned sc[PER / 2];
  fetch_scales(0, sc);
#pragma unroll
  for (int b = 0; b < B; ++b) fetch_x(0, b, xs[b]);
#pragma unroll
  for (int step = 1; step < STEPS; ++step) {
    if (step >= steps) break;
    fetch_scales(step, later_scales[step]);
#pragma unroll
    for (int b = 0; b < B; ++b) fetch_x(step, b, later[step][b]);
  }
#pragma unroll
  for (int j = 0; j < KB; ++j) fetch_w(0, j);
  __builtin_amdgcn_sched_barrier(0);

  // Digits hold all sizes, if none is beyond NF4_GATE times the run's mean. Else they hold up to
  // 128 times a mean of sizes clipped at itself (twice the mean, clipped, again and again while
  // that at least halves it), which a few sizes can't move however large.
  const float share = 1.f / (KB * 128 * steps);
  float mean[B], top[B], next[B];
  auto add_sizes = [&](const unsigned* s, int b, const float* v, bool clip) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const float size = fabsf(v[i] * __uint_as_float(i & 1 ? s[i / 2] & 0xFFFF0000u : s[i / 2] << 16));
      if (clip) {
        next[b] += fminf(size, mean[b]) * share;  // NaNs are clipped, too
      } else {
        mean[b] += size;
        top[b] = fmaxf(top[b], size);
      }
    }
  };
  auto add_all = [&](bool clip) {
#pragma unroll
    for (int b = 0; b < B; ++b) add_sizes(sc, b, xs[b], clip);
#pragma unroll
    for (int step = 1; step < STEPS; ++step) {
      if (step >= steps) break;
#pragma unroll
      for (int b = 0; b < B; ++b) add_sizes(later_scales[step], b, later[step][b], clip);
    }
  };
#pragma unroll
  for (int b = 0; b < B; ++b) mean[b] = top[b] = 0.f;
  add_all(false);
  unsigned most[B];  // bits of the largest size that digits hold
  bool loud = false;
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const unsigned sum = wave_all<false>(mean[b]) & 0x7FFFFFFFu;
    mean[b] = __uint_as_float(min(sum, NF4_FINITE)) * share;
    most[b] = wave_all<true>(top[b]);
    loud |= most[b] > __float_as_uint(mean[b] * NF4_GATE) || sum > NF4_FINITE;  // the latter: infinities, NaNs
  }
  if (__builtin_expect(loud, 0)) {
#pragma unroll
    for (int b = 0; b < B; ++b) red[(wave * B + b) * 64 + lane] = 0.f;
    for (bool more = true; more;) {
#pragma unroll
      for (int b = 0; b < B; ++b) next[b] = 0.f;
      add_all(true);
      more = false;
#pragma unroll
      for (int b = 0; b < B; ++b) {
        next[b] = __uint_as_float(wave_all<false>(next[b])) * 2.f;
        if (next[b] < mean[b] * 0.5f) {  // uniform
          mean[b] = next[b];
          more = true;
        }
      }
    }
#pragma unroll
    for (int b = 0; b < B; ++b) most[b] = min(__float_as_uint(mean[b] * 128.f), NF4_FINITE);
    wave_fence();
  }
  // takes what digits don't hold out of a step's inputs: in 32-bit floats, a column per lane
  auto strip = [&](int step) {
    unsigned over = 0;
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const float v = xs[b][i] * __uint_as_float(i & 1 ? sc[i / 2] & 0xFFFF0000u : sc[i / 2] << 16);
        if ((__float_as_uint(v) & 0x7FFFFFFFu) > most[b]) {
          xs[b][i] = 0.f;
          over |= 1u << (b * PER + i);
        }
      }
    const unsigned char* bytes = reinterpret_cast<const unsigned char*>(tiles + ((size_t)nb * kb_stride + kb0) * 256);
    for (unsigned long long lanes = __ballot(over != 0); lanes; lanes &= lanes - 1) {
      const int from = __ffsll((long long)lanes) - 1;
      for (unsigned left = __builtin_amdgcn_readlane((int)over, from); left; left &= left - 1) {
        const int bit = __ffs((int)left) - 1, b = bit / PER, i = step * KB * 128 + from * PER + bit % PER;
        const int at = i % 16, half = i % 128 / 64;
        const int byte = (((i / 128) * 4 + lane / 16) * 64 + i % 64 / 16 * 16 + lane % 16) * 16 + half * 8 + at / 8 * 4 + at % 4;
        const float level = NF4_TILE_LEVELS[at & 4 ? bytes[byte] >> 4 : bytes[byte] & 15];
        const float weight = level * bf16_to_f32(scales[((size_t)nb * kb_stride + kb0) * 128 + i]);
        float* sum = &red[(wave * B + b) * 64 + lane];
        *sum = fmaf(weight, x[(size_t)b * x_stride + kb0 * 128 + i], *sum);
      }
    }
  };
  float unit[B], factor[B];  // the scaled inputs' last place, and one over it
#pragma unroll
  for (int b = 0; b < B; ++b) {
    // below 2^(e - 126), times 2^(156 - e)
    const unsigned up = min(283u - (most[b] >> 23), 253u);
    factor[b] = __uint_as_float(up << 23);
    unit[b] = __uint_as_float((254u - up) << 23);
  }

  // Digits of an input's rows are neighbours; loads that transpose bytes make them columns. A lane has 8 slots of 16
  // bytes, turned by half its number, so that 16 lanes that write the same one use all banks.
  unsigned char* const mine = digits[wave];
  auto slot_at = [](int block, int slot) { return block * 128 + ((slot + (block >> 1)) & 7) * 16; };
  auto put = [&](int i, const unsigned* q) {  // digits of this lane's i-th input
    if constexpr (WIDE) {
      *reinterpret_cast<u32x4*>(mine + slot_at(lane, 2 * i)) = u32x4{q[0], q[1], q[2], q[3]};
      *reinterpret_cast<u32x4*>(mine + slot_at(lane, 2 * i + 1)) =
          u32x4{q[4], B > 5 ? q[B > 5 ? 5 : 0] : 0u, B > 6 ? q[B > 6 ? 6 : 0] : 0u, B > 7 ? q[B > 7 ? 7 : 0] : 0u};
    } else {
      *reinterpret_cast<u32x4*>(mine + slot_at(lane, i)) =
          u32x4{q[0], B > 1 ? q[B > 1 ? 1 : 0] : 0u, B > 2 ? q[B > 2 ? 2 : 0] : 0u, B > 3 ? q[B > 3 ? 3 : 0] : 0u};
    }
  };
  // a lane's column of 16 inputs: those of tile j, half, and run hi, or (h * 2 + run), in two loads
  int from[WIDE ? 4 : 2];
  if constexpr (WIDE) {
    const int row = col / 2, h = hi >> 1;
#pragma unroll
    for (int i = 0; i < 4; ++i)  // 2 run + which of the loads
      from[i] = h * 8 * 128 + row / 4 * 128 + ((row % 4 * 2 + (hi & 1) + h * 4 + i) & 7) * 16 + (col & 1) * 8;
  } else {
    const int row = col / 2;
#pragma unroll
    for (int i = 0; i < 2; ++i)  // half
      from[i] = hi * 2 * 128 + ((row + hi + i * 4) & 7) * 16 + (col & 1) * 8;
  }
  auto column = [&](int j, int half, int run) {
    using lds_two = __attribute__((address_space(3))) i32x2;
    i32x2 v[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int at = WIDE ? from[2 * run + i] + (j * 32 + half * 16 + run * 4 + i * 2) * 128 : from[half] + (j * 16 + half * 8 + i) * 128;
      v[i] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_two*)(mine + at));
    }
    return i32x4{v[0][0], v[0][1], v[1][0], v[1][1]};
  };
  // the digits of four codes in a byte each, or what makes them up
  auto look_up = [&](unsigned w0, unsigned w1, int p, i32x4& a, i32x4& b) {
    constexpr auto& table = SUMMED ? NF4_SUMMANDS : NF4_DIGITS;
    // codes 0-7 select below 8; the others do with bit 3 turned
    const unsigned lo[4] = {w0 & 0x0F0F0F0Fu, (w0 >> 4) & 0x0F0F0F0Fu, w1 & 0x0F0F0F0Fu, (w1 >> 4) & 0x0F0F0F0Fu};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[i] = (int)__builtin_amdgcn_perm(table[p][1], table[p][0], lo[i]);
      b[i] = (int)__builtin_amdgcn_perm(table[p][3], table[p][2], lo[i] ^ 0x08080808u);
    }
  };

  using sums = __attribute__((ext_vector_type(WIDE ? 16 : 4))) int;
  constexpr int G = WIDE ? 2 : 4;  // runs of 32 or 16 columns
  sums acc[G][3];
#pragma unroll
  for (int c = 0; c < G; ++c)
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int r = 0; r < (WIDE ? 16 : 4); ++r) acc[c][p][r] = 0;

  for (int step = 0; step < steps; ++step) {
    if (__builtin_expect(loud, 0)) strip(step);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const float s = __uint_as_float(i & 1 ? sc[i / 2] & 0xFFFF0000u : sc[i / 2] << 16);
      unsigned q[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const float v = xs[b][i] * s;
        q[b] = ((unsigned)(int)rintf(v * factor[b]) + 0x00808080u) ^ 0x00808080u;
      }
      put(i, q);
    }
    wave_fence();
    const int beyond = step + 1 < steps ? 0 : NF4_BEYOND;
    if (LONG) {
      fetch_scales(step + 1, sc, beyond);
#pragma unroll
      for (int b = 0; b < B; ++b) fetch_x(step + 1, b, xs[b], beyond);
    }
#pragma unroll
    for (int j = 0; j < KB; ++j) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int run = 0; run < (WIDE ? 2 : 1); ++run) {
          const i32x4 xd = column(j, half, run);
#pragma unroll
          for (int c = 0; c < G; ++c) {
            const u32x4& codes = w[j][WIDE ? 2 * c + run : c];
#pragma unroll
            for (int p = 0; p < 3; ++p) {
              i32x4 a, b;
              look_up(half ? codes.z : codes.x, half ? codes.w : codes.y, p, a, b);
              if constexpr (WIDE) {
                acc[c][p] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a ^ b, xd, acc[c][p], 0, 0, 0);
              } else {
                acc[c][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, xd, acc[c][p], 0, 0, 0);
                acc[c][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, xd, acc[c][p], 0, 0, 0);
              }
            }
            if constexpr (!WIDE)
#pragma unroll
              for (int i = 0; i < 6; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
              }
          }
        }
      }
      if (LONG) fetch_w(step + 1, j, beyond);
    }
    wave_fence();
  }

  // this lane's column of digits is that of a row and, in it, of the digit n % 4; it has four neighbouring
  // columns of weights at a time
  const int n = WIDE ? lane & 31 : col, row = n / 4, first = WIDE ? (hi >> 1) * 4 : hi * 4;
  float last = 0.f;
#pragma unroll
  for (int b = 0; b < B; ++b) last = row == b ? unit[b] : last;
  const float place = __uint_as_float((127u + 8u * (n & 3)) << 23) * NF4_UNIT;
#pragma unroll
  for (int c = 0; c < G; ++c)
#pragma unroll
    for (int f = 0; f < (WIDE ? 4 : 1); ++f) {
      float4v v;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float sum = fmaf((float)acc[c][2][4 * f + r], 65536.f, fmaf((float)acc[c][1][4 * f + r], 256.f, (float)acc[c][0][4 * f + r]));
        v[r] = quad_sum(sum * place) * last;
      }
      if ((n & 3) == 0 && row < B) {
        float4v* sum = reinterpret_cast<float4v*>(&red[(wave * B + row) * 64 + c * (64 / G) + f * 8 + first]);
        *sum = loud ? *sum + v : v;
      }
    }
  __syncthreads();
  for (int i = tid; i < B * 64; i += 256) {
    const float sum = (red[i] + red[B * 64 + i]) + (red[2 * B * 64 + i] + red[3 * B * 64 + i]);
    const size_t row = sel ? (size_t)blockIdx.y * gridDim.z + blockIdx.z : (size_t)blockIdx.y * B + i / 64;
    partials[row * out_dim + nb * 64 + i % 64] = sum;
  }
}

// ------------------------------------------------------------ packing

// one thread per 16 bytes of a tile
__global__ void nf4_tile_kernel(
    const unsigned char* __restrict__ packed,   // [in, out/2]
    const unsigned short* __restrict__ absmax,  // [in, out/64]
    uint4* __restrict__ tiles, unsigned short* __restrict__ scales, int in_dim, int out_dim, int n_kb) {
  const size_t at = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t n = (size_t)(out_dim / 64) * n_kb;
  if (at < n * 256) {
    const int lane = at % 64, c = at / 64 % 4, kb = at / 256 % n_kb;
    const size_t nb = at / 256 / n_kb;
    const size_t column = nb * 64 + c * 16 + lane % 16;
    unsigned words[4] = {0u, 0u, 0u, 0u};
    for (int i = 0; i < 32; ++i) {
      const int k = kb * 128 + i / 16 * 64 + lane / 16 * 16 + i % 16;
      unsigned code = 7u;  // 0
      if (k < in_dim) {
        const unsigned char byte = packed[((size_t)k * out_dim + column) / 2];
        code = column & 1 ? byte >> 4 : byte & 15;
      }
      words[i / 8] |= code << ((i & 3) * 8 + (i & 4));
    }
    tiles[at] = uint4{words[0], words[1], words[2], words[3]};
  }
  if (at < n * 128) {
    const int k = at % ((size_t)n_kb * 128);
    const size_t nb = at / ((size_t)n_kb * 128);
    scales[at] = k < in_dim ? absmax[(size_t)k * (out_dim / 64) + nb] : (unsigned short)0;
  }
}

// A tile per workgroup: dense[k, n] = bf16(level * scale), 128 bytes of a row at a time
__global__ __launch_bounds__(256) void nf4_untile_kernel(
    const uint4* __restrict__ tiles, const unsigned short* __restrict__ scales, unsigned short* __restrict__ dense,
    int in_dim, int out_dim, int n_kb) {
  __shared__ float levels[16];
  __shared__ unsigned short scale[128];
  __shared__ unsigned short tile[128][64 + 2];
  const int tid = threadIdx.x, lane = tid & 63, c = tid >> 6;
  const int kb = blockIdx.x % n_kb, nb = blockIdx.x / n_kb;
  if (tid < 16) levels[tid] = NF4_TILE_LEVELS[tid];
  if (tid < 128) scale[tid] = scales[((size_t)nb * n_kb + kb) * 128 + tid];
  const uint4 w = tiles[(size_t)blockIdx.x * 256 + tid];
  const unsigned words[4] = {w.x, w.y, w.z, w.w};
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const int k = i / 16 * 64 + lane / 16 * 16 + i % 16;
    const unsigned code = (words[i / 8] >> ((i & 3) * 8 + (i & 4))) & 15u;
    tile[k][c * 16 + lane % 16] = f32_to_bf16(levels[code] * bf16_to_f32(scale[k]));
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int k = i * 8 + tid / 32, n = tid % 32 * 2;
    if (kb * 128 + k < in_dim)
      *reinterpret_cast<unsigned*>(dense + (size_t)(kb * 128 + k) * out_dim + nb * 64 + n) =
          *reinterpret_cast<const unsigned*>(&tile[k][n]);
  }
}

// ------------------------------------------------------------------- host

// packed [in, out/2], absmax [in, out/64] -> (tiles, scales); [E, ...] for stacked experts
std::vector<torch::Tensor> nf4_tile(torch::Tensor packed, torch::Tensor absmax) {
  TORCH_CHECK(packed.is_cuda() && packed.dtype() == torch::kUInt8 && packed.dim() == 2 && packed.is_contiguous());
  TORCH_CHECK(absmax.is_cuda() && absmax.dtype() == torch::kBFloat16 && absmax.is_contiguous());
  const long in_dim = packed.size(0), out_dim = packed.size(1) * 2;
  TORCH_CHECK(in_dim > 0 && out_dim % 64 == 0 && absmax.dim() == 2 && absmax.size(0) == in_dim &&
              absmax.size(1) == out_dim / 64);
  const long n_kb = (in_dim + 127) / 128, nb = out_dim / 64;
  auto tiles = torch::empty({nb, n_kb, 4, 64, 16}, packed.options());
  auto scales = torch::empty({nb, n_kb * 128}, absmax.options());
  const long threads = nb * n_kb * 256;
  TORCH_CHECK(threads / 256 < (1L << 31));
  nf4_tile_kernel<<<threads / 256, 256, 0, at::cuda::getCurrentCUDAStream()>>>(
      packed.data_ptr<unsigned char>(), reinterpret_cast<const unsigned short*>(absmax.data_ptr()),
      reinterpret_cast<uint4*>(tiles.data_ptr()), reinterpret_cast<unsigned short*>(scales.data_ptr()), (int)in_dim,
      (int)out_dim, (int)n_kb);
  HIP_CHECK_LAST();
  return {tiles, scales};
}

static void check_tiles(const torch::Tensor& tiles, const torch::Tensor& scales, int64_t in_dim, int lead) {
  TORCH_CHECK(tiles.is_cuda() && tiles.dtype() == torch::kUInt8 && tiles.dim() == 5 + lead && tiles.is_contiguous());
  TORCH_CHECK(scales.is_cuda() && scales.dtype() == torch::kBFloat16 && scales.dim() == 2 + lead && scales.is_contiguous());
  const long nb = tiles.size(lead), n_kb = tiles.size(lead + 1);
  TORCH_CHECK(tiles.size(lead + 2) == 4 && tiles.size(lead + 3) == 64 && tiles.size(lead + 4) == 16);
  TORCH_CHECK(scales.size(lead) == nb && scales.size(lead + 1) == n_kb * 128);
  TORCH_CHECK(lead == 0 || scales.size(0) == tiles.size(0));
  TORCH_CHECK(in_dim > 0 && (in_dim + 127) / 128 == n_kb, "tiles of other inputs");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(tiles.data_ptr()) % 16 == 0 && reinterpret_cast<uintptr_t>(scales.data_ptr()) % 4 == 0);
}

torch::Tensor nf4_untile(torch::Tensor tiles, torch::Tensor scales, int64_t in_dim) {
  check_tiles(tiles, scales, in_dim, 0);
  const long nb = tiles.size(0), n_kb = tiles.size(1);
  auto dense = torch::empty({in_dim, nb * 64}, scales.options());
  nf4_untile_kernel<<<nb * n_kb, 256, 0, at::cuda::getCurrentCUDAStream()>>>(
      reinterpret_cast<const uint4*>(tiles.data_ptr()), reinterpret_cast<const unsigned short*>(scales.data_ptr()),
      reinterpret_cast<unsigned short*>(dense.data_ptr()), (int)in_dim, (int)(nb * 64), (int)n_kb);
  HIP_CHECK_LAST();
  return dense;
}

// sel: [rows] experts or null; returns [splits, rows, out]
static torch::Tensor launch_nf4_tiles(
    const torch::Tensor& tiles, const torch::Tensor& scales, int64_t in_dim, const torch::Tensor& x,
    const torch::Tensor* sel, int64_t k_per_tok, torch::Tensor workspace) {
  const int lead = sel ? 1 : 0;
  const long nb = tiles.size(lead), n_kb = tiles.size(lead + 1), out_dim = nb * 64;
  TORCH_CHECK(x.is_cuda() && x.dtype() == torch::kFloat32 && x.dim() == 2 && x.is_contiguous() && x.size(1) == in_dim);
  const int batch = sel ? 1 : (int)x.size(0);
  const long rows = sel ? sel->numel() : batch, z = sel ? rows : 1;
  TORCH_CHECK(batch >= 1 && batch <= 8, "NF4 products of few rows take at most 8");
  const int kb = batch <= 4 ? 4 : 2;
  // longer runs combine their sums once, but only where enough waves remain
  const long units = nb * z * ((n_kb + kb - 1) / kb);
  long steps = 1;
  while (batch > 4 && steps < 4 && units / (2 * steps) >= 2048) steps *= 2;
  const long splits = (n_kb + 4 * kb * steps - 1) / (4 * kb * steps);
  TORCH_CHECK(workspace.numel() == 0 || (workspace.is_cuda() && workspace.dtype() == torch::kFloat32));
  torch::Tensor partials = workspace.numel() >= splits * rows * out_dim
                               ? workspace.view(-1).narrow(0, 0, splits * rows * out_dim).view({splits, rows, out_dim})
                               : torch::empty({splits, rows, out_dim}, x.options());
  if (z == 0) return partials;
  const bool by4 = in_dim % 4 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
  auto stream = at::cuda::getCurrentCUDAStream();
  for (long first = 0; first < n_kb; first += NF4_LAUNCH) {
    const long run = std::min<long>(n_kb - first, NF4_LAUNCH), inputs = std::min<long>(in_dim - first * 128, NF4_LAUNCH * 128);
    const dim3 grid(nb, (run + 4 * kb * steps - 1) / (4 * kb * steps), z);
#define NF4_TILES(B, KB)                                                                                            \
  gemv_nf4_tiles_kernel<B, KB><<<grid, 256, 0, stream>>>(                                                           \
      reinterpret_cast<const uint4*>(tiles.data_ptr()) + first * 256,                                               \
      reinterpret_cast<const unsigned short*>(scales.data_ptr()) + first * 128, x.data_ptr<float>() + first * 128,  \
      sel ? sel->data_ptr<int>() : nullptr, partials.data_ptr<float>() + first / (4 * kb * steps) * rows * out_dim, \
      (int)inputs, (int)out_dim, (int)run, (int)steps, (int)k_per_tok, sel ? (int)tiles.size(0) : 1, by4,           \
      (int)in_dim, (int)n_kb)
    switch (batch) {
      case 1: NF4_TILES(1, 4); break;
      case 2: NF4_TILES(2, 4); break;
      case 3: NF4_TILES(3, 4); break;
      case 4: NF4_TILES(4, 4); break;
      case 5: NF4_TILES(5, 2); break;
      case 6: NF4_TILES(6, 2); break;
      case 7: NF4_TILES(7, 2); break;
      case 8: NF4_TILES(8, 2); break;
    }
#undef NF4_TILES
    HIP_CHECK_LAST();
  }
  return partials;
}

torch::Tensor gemv_nf4_tiles(
    torch::Tensor tiles, torch::Tensor scales, int64_t in_dim,
    torch::Tensor x,  // [batch, in] f32
    torch::Tensor workspace, c10::optional<torch::Tensor> residual, int64_t epilogue,
    c10::optional<torch::Tensor> bias) {  // epilogue < 0: the partial sums [splits, batch, out]
  check_tiles(tiles, scales, in_dim, 0);
  auto partials = launch_nf4_tiles(tiles, scales, in_dim, x, nullptr, 1, workspace);
  if (epilogue < 0) return partials;
  return launch_gemv_reduce(partials, residual, bias, (int)partials.size(0), (int)partials.size(1),
                            (int)partials.size(2), (int)epilogue, x.options(), scales.options());
}

torch::Tensor gemv_nf4_tiles_moe(
    torch::Tensor tiles, torch::Tensor scales, int64_t in_dim,
    torch::Tensor x,    // [B, in] f32
    torch::Tensor sel,  // [R] int32, R = B * k_per_tok
    int64_t k_per_tok, torch::Tensor workspace, int64_t epilogue) {
  check_tiles(tiles, scales, in_dim, 1);
  TORCH_CHECK(sel.is_cuda() && sel.dtype() == torch::kInt32 && sel.is_contiguous());
  const long rows = sel.numel();
  TORCH_CHECK(x.dim() == 2 && rows == x.size(0) * k_per_tok);
  TORCH_CHECK(rows <= 16, "moe gemv supports batch*k <= 16");
  auto partials = launch_nf4_tiles(tiles, scales, in_dim, x, &sel, k_per_tok, workspace);
  if (epilogue < 0) return partials;
  return launch_gemv_reduce(partials, c10::nullopt, c10::nullopt, (int)partials.size(0), (int)rows,
                            (int)partials.size(2), (int)epilogue, x.options(), scales.options());
}
