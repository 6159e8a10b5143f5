// Products of 2 to some hundreds of rows with rounded weights (see gemm_block_q.hip): panels of
// 16 TM rows of x against 64 TN columns of W.  The waves lie along the columns, so that every
// weight of a panel is widened by one wave only, once for all its rows.
//
// x and W reach LDS without registers, STAGES tiles of 64 inputs deep.  The barrier lies in the
// middle of a tile's products, behind which the next tile may be read: its first fragments and
// weights are on their way or widened before the tile begins, and a tile's loads are asked for
// one by one between the products (a burst keeps all waves from them).  Neighbouring columns
// start a tile of K apart (4096 x 4096, 301 rows 20.0 -> 18.8 us).
//
// In large panels a pair of weights is widened behind each product of the step before: one more
// instruction hides behind v_mfma_f32_16x16x32_bf16 (16 clocks), each further one adds four to a
// lone wave's time (28672 x 4096, 301 rows: 80 -> 77 us, and 2 % over four layers under sustained load;
// 96 x 128, two a CU, 4096 x 14336, 700 rows 107 | 110, as before.  Products of 32 x
// 32, which hide five, take 69 us alone but more power: the clock falls from 2360 to 2180 MHz, four
// layers 718 | 727).  LDS serves 16-byte reads sixteen lanes at a time, half of them of one quarter of
// the wave and half of the next (0..3, 12..15, 20..27 | 4..11, 16..19, 28..31): chunks lie so that these
// are in different banks (half of all LDS cycles were conflicts).
//
// 4 bits: a nibble less its offset becomes a float in one instruction (v_cvt_off_f32_i4, of two's
// complement), whose upper half is all of it, so that there is no offset to take from the sums (8 + n/2
// by bit patterns, cheaper by a third, needs the sum of x of every row and group).  Sums of a group of 128
// inputs are apart: its first product begins them and a row late each is multiplied by its column's
// scale into the whole ones, four instructions for every four products of 16 x 16 x 32, beside those
// that widen.  With two workgroups a CU they hide behind the other's products: 28672 x 4096, 196
// rows 0.69 PFLOP/s, 900 rows 0.88 (int8 0.76, 0.98).  W's rows of a tile are 32 bytes.
//
// Gated, half of a wave's columns are gates and half what they multiply, and the launch that did
// that (6 us at 301 x 28672) with its reads of the product falls away.
#pragma once

#include <type_traits>

#include "block_gemm.h"
#include "moe_tiles.h"

namespace gemm_panel {

using block_gemm::bf16x8_t;
using block_gemm::f32x4_t;

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2_t;
// scales start at any float
typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any_t;

constexpr int kDepth = 64;    // inputs of a tile
constexpr int kWaves = 4;     // along N

// A wave's loads of n tiles, of `each` and, for 4 bits, the scales of a group of two with its
// first; half: of the first tile
template <int QB> constexpr int loads_of(int each, int half, int n) {
  return n * each + (QB == 4 ? (n + 1 - half % 2) / 2 : 0);
}

// The low nibble of byte d as a whole number of two's complement, over 16.  (VALU only, and all of
// the result's bits are written: nothing for the compiler to wait for.)
DEVINLINE unsigned nibble(unsigned v, int d) {
  unsigned f;
#define CVT(B)                                                                      \
  asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_" #B \
      : "=v"(f) : "v"(v))
  if (d == 0) CVT(0);
  else if (d == 1) CVT(1);
  else if (d == 2) CVT(2);
  else CVT(3);
#undef CVT
  return f;
}

// grid (tiles of y, parts of K); part [parts, M, N] (gridDim.y > 1); depth: inputs of a part (4
// bits: whole groups of 128)
// PER_CU: workgroups that share a CU.  GATED: N outputs of 2 N rows of W, K in one part.
template <int QB, int TM, int TN, int STAGES, int PER_CU, bool GATED>
__global__ __launch_bounds__(64 * kWaves, PER_CU) void gemm_panel_q_kernel(
    __hip_bfloat16* __restrict__ y,         // [M, N]
    float* __restrict__ part,
    const __hip_bfloat16* __restrict__ x,   // [M, K]
    const unsigned char* __restrict__ w,    // int8 [N, K] | [2 N, K]; 4 bits [.., K / 2]
    const float* __restrict__ scale,        // [N] | [2 N]; 4 bits [.., K / 128]
    const int M, const int N, const int K, const int depth) {
  constexpr int BM = TM * 16, BN = TN * 16 * kWaves;
  constexpr int W_ROW = kDepth * QB / 8, WL = W_ROW / 16;   // bytes and lanes of a W row
  constexpr int X_BYTES = BM * kDepth * 2, W_BYTES = BN * W_ROW;
  constexpr int STAGE = X_BYTES + W_BYTES + (QB == 4 ? BN * 4 : 0);
  constexpr int X_LOADS = BM / 8, W_LOADS = W_BYTES / 1024;   // 1 KB each
  constexpr int X_PASS = (X_LOADS + kWaves - 1) / kWaves;
  constexpr int W_PASS = (W_LOADS + kWaves - 1) / kWaves;
  constexpr int LOADS = X_PASS + W_PASS;
  // fragments of x on their way; those of the next tile are asked for behind the barrier
  constexpr int AHEAD = TM < 3 ? TM : 3;
  constexpr bool SPREAD = TM >= 8;        // widening over the products
  // results of a wave and of a panel; one tile a wave has eight gates and eight of the others
  constexpr int WIDE = TN * (GATED ? 8 : 16), COLS = WIDE * kWaves;
  constexpr bool HALVES = GATED && TN == 1;
  constexpr int OUT = GATED && !HALVES ? TN / 2 : TN;
  static_assert(!GATED || HALVES || TN % 2 == 0, "as many gates");
  static_assert(TM >= TN && TM >= AHEAD && STAGES >= 3, "what a tile's products hide");
  static_assert(STAGES * STAGE * PER_CU <= 160 * 1024, "LDS of a CU");
  __shared__ __align__(16) char lds[STAGES * STAGE];

  // neighbours in a run of blocks that one XCD gets share their columns of W
  const int m_tiles = (M + BM - 1) / BM, blocks = m_tiles * (N / COLS);
  const int per_xcd = (blocks + 7) / 8, slot = blockIdx.x / 8;
  const int id = (blockIdx.x % 8) * per_xcd + slot;
  if (slot >= per_xcd || id >= blocks) return;
  const int k0 = blockIdx.y * depth;
  const int m0 = id % m_tiles * BM, n0 = id / m_tiles * COLS;
  const int tiles = min(depth, K - k0) / kDepth;
  const int start = QB == 4 ? id / m_tiles % (tiles / 2) * 2 : id / m_tiles % tiles;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, quad = lane >> 4;

  // (4 bits: the reads of a wave are one run of bytes)
  auto w_turn = [](int r) { return QB == 4 ? 0 : SPREAD ? -(r / 4) & 3 : r / 4 % 4; };
  // Pass p of the waves' over a tile's loads.  (Where the last has fewer than waves some are made twice: all
  // waves wait alike.)  Only there is a remainder taken past 64 rows: other places are the wave's own
  // and a literal.  With remainders everywhere the loop of 160 x 256 had 282 instructions, now 271, each four
  // clocks of a wave alone on its SIMD: four layers of llama-3-8b in int8, 150 rows 506 -> 492 us, 301
  // rows 716 -> 706; of 80 x 64, 4096 x 4096, 257 rows 21.0 -> 19.1.  (Panels of fewer rows, of which two
  // share a SIMD, gain nothing: 40 rows 326 as they are, 330.)
  auto pass = [&](int p, int loads) {
    const int at = p * kWaves + wave;
    return TM > 4 && (p + 1) * kWaves <= loads ? at : at % loads;
  };
  // (rows of a panel are found by 32 bits, see gemm_panel_plan)
  unsigned x_off[X_PASS], w_off[W_PASS];
#pragma unroll
  for (int p = 0; p < X_PASS; ++p) {
    const int r = pass(p, X_LOADS) * 8 + lane / 8;
    const int at = (lane % 8) ^ (r / 2 % 8);   // large: of the chunks 0 2 4 6 1 3 5 7
    x_off[p] = (unsigned)min(r, M - 1 - m0) * (K * 2u) + (SPREAD ? at % 4 * 2 + at / 4 : at) * 16;
  }
  auto w_row = [&](int r) {   // of W from n0 on, for row r of the panel's
    const int own = r / (TN * 16), in = r % (TN * 16);
    return (unsigned)(in / WIDE * N + own * WIDE + in % WIDE);
  };
#pragma unroll
  for (int p = 0; p < W_PASS; ++p) {
    const int r = pass(p, W_LOADS) * (64 / WL) + lane / WL;
    w_off[p] = w_row(r) * (unsigned)(K * QB / 8) + ((lane % WL) ^ w_turn(r)) * 16;
  }
  const auto x_from = block_gemm::resource(x + (long)m0 * K + k0);
  const auto w_from = block_gemm::resource(w + ((long)n0 * K + k0) * QB / 8);
  unsigned s_off = 0;
  if constexpr (QB == 4) s_off = w_row(wave % TN * 64 + lane) * (unsigned)(K / 128 * 4);
  const auto s_from =
      block_gemm::resource(QB == 4 ? scale + (long)n0 * (K / 128) + k0 / 128 : scale);
  // load p of a tile (past the last tile it is the last one again) to the buffer of which `own` is the
  // wave's first KB: places are that and a literal, or a register where a remainder is taken
  auto load = [&](int& own, int tile, int p) {
    tile = min(tile, tiles - 1) + start;
    if (tile >= tiles) tile -= tiles;
    // Added as the load is made, in one instruction: where loads are many the compiler adds all ahead and
    // copies each.  (Elsewhere it does well alone, and keeping the order costs: 4 bits 28672 x 4096, 129
    // rows 47.8 us, 59.6 with it; int8 4096 x 4096, 196 rows 18.9, 20.9)
    if constexpr (QB == 8 && TN == 4) asm volatile("" : "+s"(own));
    auto place = [&](int q, int loads) { return lds + own + (pass(q, loads) - wave) * 1024; };
    if (p < X_PASS)
      block_gemm::load_lds(place(p, X_LOADS), x_from, x_off[p], tile * (kDepth * 2));
    else if (p < LOADS)
      block_gemm::load_lds(place(p - X_PASS, W_LOADS) + X_BYTES, w_from,
                           w_off[p < LOADS ? p - X_PASS : 0], tile * W_ROW);
    else
      block_gemm::load_lds4(lds + own + (X_BYTES + W_BYTES + wave % TN * 256 - wave * 1024), s_from,
                            s_off, tile / 2 * 4);
  };

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_t{};
  // 4 bits: sums of a group, ahead of its scales
  f32x4_t part_sum[QB == 4 ? TM : 1][QB == 4 ? TN : 1], group_scale[QB == 4 ? TN : 1];

  // A lane's 16 weights of a column (chunk quad of its row) are its inputs of two matrix steps,
  // and x is read to match.
  auto x_frag = [&](const char* at, int s, int i) {
    const int r = i * 16 + col;
    return *reinterpret_cast<const bf16x8_t*>(at + r * (kDepth * 2) +
                                              ((SPREAD ? s * 4 + quad : quad * 2 + s) ^
                                               (r / 2 % 8)) * 16);
  };
  auto w_chunk = [&](const char* at, int j) {
    const int r = (wave * TN + j) * 16 + col;
    if constexpr (QB == 4)
      return *reinterpret_cast<const u32x2_t*>(at + X_BYTES + r * W_ROW + quad * 8);
    else
      return *reinterpret_cast<const u32x4_t*>(at + X_BYTES + r * W_ROW +
                                               (quad ^ w_turn(r)) * 16);
  };
  using Chunk = decltype(w_chunk(lds, 0));
  auto unpack = [&](const Chunk& c, int s, int d) {   // pair d of a column's weights of step s
    if constexpr (QB == 4) {
      const unsigned eight = c[s] ^ 0x88888888u;   // n - 8 in two's complement
      return __builtin_amdgcn_perm(nibble(eight >> 4, d), nibble(eight, d), 0x07060302);
    }
    const unsigned four = c[2 * s + d / 2] >> (d % 2 * 16);
    const float a = (float)(signed char)(four & 0xff);
    const float b = (float)(signed char)((four >> 8) & 0xff);
    // whole numbers of 8 bits: the upper half of the float is all of it
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
  };

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) {
    int own = s * STAGE + wave * 1024;
#pragma unroll
    for (int p = 0; p < loads_of<QB>(LOADS, s, 1); ++p) load(own, s, p);
  }
  block_gemm::wait_loads<loads_of<QB>(LOADS, 1, STAGES - 2)>();
  block_gemm::meet();
  Chunk c[TN];
  u32x4_t wf[2][TN];
  bf16x8_t xf[AHEAD];
#pragma unroll
  for (int j = 0; j < TN; ++j) c[j] = w_chunk(lds, j);
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int d = 0; d < 4; ++d) wf[0][j][d] = unpack(c[j], 0, d);
#pragma unroll
  for (int q = 0; q < AHEAD; ++q) xf[q] = x_frag(lds, q / TM, q % TM);

  auto finish = [&](int i, int j) {
    if constexpr (QB == 4) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[i][j][r] = __builtin_fmaf(group_scale[j][r], part_sum[i][j][r], acc[i][j][r]);
    }
  };
  int buf = 0;
  auto turn = [&](int t, auto which) {
    constexpr int HALF = decltype(which)::value;   // 4 bits: of a group
    const int after = buf + 1 == STAGES ? 0 : buf + 1, before = buf == 0 ? STAGES - 1 : buf - 1;
    const char* here = lds + buf * STAGE;
    const char* there = lds + after * STAGE;
    int own = before * STAGE + wave * 1024;   // of the tile that is asked for
    bf16x8_t xr[2 * TM + AHEAD];
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) xr[q] = xf[q];
#pragma unroll
    for (int q = 0; q < 2 * TM; ++q) {   // 16 rows of x and 32 inputs at a time
      const int s = q / TM, i = q % TM;
      if (q == TM) {
        // the next tile is here, and all have read the one before this one
        block_gemm::wait_loads<loads_of<QB>(LOADS, HALF, STAGES - 3)>();
        block_gemm::meet();
#pragma unroll
        for (int j = 0; j < TN; ++j) c[j] = w_chunk(there, j);
      }
      constexpr int ASKED = loads_of<QB>(LOADS, HALF + STAGES - 1, 1);
#pragma unroll
      for (int p = 0; p < ASKED; ++p)
        if (s == 1 && p * TM / ASKED == i) load(own, t + STAGES - 1, p);
      if constexpr (QB == 4 && HALF == 0)
        if (q == 0)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            group_scale[j] = *reinterpret_cast<const f32x4_t*>(
                here + X_BYTES + W_BYTES + ((wave * TN + j) * 16 + quad * 4) * 4);
      const int f = q + AHEAD;
      xr[f] = f < 2 * TM ? x_frag(here, f / TM, f % TM)
                         : x_frag(there, (f - 2 * TM) / TM, (f - 2 * TM) % TM);
      // the weights of the next step, a column at a time or a pair behind each product (of the
      // next tile two rows of products late: its weights are on their way)
      constexpr int PAIRS = 4 * TN, LATE = 2 * TN;
      const int room = s == 0 ? TM * TN : TM * TN - LATE;
      if (!SPREAD && (s == 0 ? i < TN : i >= TM - TN)) {
        const int j = s == 0 ? i : i - (TM - TN);
#pragma unroll
        for (int d = 0; d < 4; ++d) wf[1 - s][j][d] = unpack(c[j], 1 - s, d);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (QB == 4) {
          part_sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, wf[s][j]), xr[q],
              HALF == 0 && s == 0 ? f32x4_t{} : part_sum[i][j], 0, 0, 0);
          // a row late: its sums are there
          if (HALF == 1 && s == 1 && i > 0) finish(i - 1, j);
        } else {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, wf[s][j]), xr[q], acc[i][j], 0, 0, 0);
        }
        const int at = i * TN + j - (s == 0 ? 0 : LATE);
        if (SPREAD && at >= 0) {
#pragma unroll
          for (int u = at * PAIRS / room; u < (at + 1) * PAIRS / room; ++u)
            wf[1 - s][u / 4][u % 4] = unpack(c[u / 4], 1 - s, u % 4);
        }
        if (SPREAD) __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) xf[q] = xr[2 * TM + q];
    if constexpr (QB == 4 && HALF == 1)
#pragma unroll
      for (int j = 0; j < TN; ++j) finish(TM - 1, j);
    buf = after;
  };
  if constexpr (QB == 4) {
    for (int t = 0; t < tiles; t += 2) {
      turn(t, std::integral_constant<int, 0>{});
      turn(t + 1, std::integral_constant<int, 1>{});
    }
  } else {
    for (int t = 0; t < tiles; ++t) turn(t, std::integral_constant<int, 0>{});
  }
  block_gemm::wait_loads<0>();   // LDS is not given back ahead of them

  const bool cut = gridDim.y > 1;
#pragma unroll
  for (int j = 0; j < OUT; ++j) {
    const int n = n0 + wave * WIDE + j * 16 + (HALVES ? quad % 2 : quad) * 4;
    f32x4_t s{16.f, 16.f, 16.f, 16.f}, su = s;   // (4 bits: what `nibble` leaves)
    if constexpr (QB == 8) {
      s = *reinterpret_cast<const f32x4_any_t*>(scale + n + (HALVES && quad >= 2 ? N : 0));
      if constexpr (GATED && !HALVES) su = *reinterpret_cast<const f32x4_any_t*>(scale + N + n);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + i * 16 + col;
      f32x4_t v;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = acc[i][j][r] * s[r];
        if constexpr (HALVES)
          v[r] = moe::finish<moe::kSilu>(v[r], __shfl_xor(v[r], 32), 0.f);
        else if constexpr (GATED)
          v[r] = moe::finish<moe::kSilu>(v[r], acc[i][OUT + j][r] * su[r], 0.f);
      }
      if (m >= M || (HALVES && quad >= 2)) continue;
      if (!GATED && cut) {
        *reinterpret_cast<f32x4_t*>(part + (blockIdx.y * (long)M + m) * N + n) = v;
      } else {
        union { __hip_bfloat16 h[4]; uint2 u; } o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o.h[r] = __float2bfloat16(v[r]);
        *reinterpret_cast<uint2*>(y + (long)m * N + n) = o.u;
      }
    }
  }
}

}  // namespace gemm_panel
