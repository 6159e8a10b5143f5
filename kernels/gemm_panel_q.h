// Products of 65 to some hundreds of rows with int8 weights (see gemm_block_q.hip): panels of
// 16 TM rows of x against 64 TN columns of W.  The waves lie along the columns, so that every
// weight of a panel is widened by one wave only, once for all its rows.
//
// x and W reach LDS without registers, STAGES tiles of 64 inputs deep.  The barrier lies in the
// middle of a tile's products, behind which the next tile may be read: its first fragments and
// weights are on their way or widened before the tile begins, and a tile's loads are asked for
// one by one between the products (a burst keeps all waves from them).  Neighbouring columns
// start a tile of K apart (4096 x 4096, 301 rows 20.0 -> 18.8 us).
#pragma once

#include "block_gemm.h"

namespace gemm_panel {

using block_gemm::bf16x8_t;
using block_gemm::f32x4_t;

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
// scales start at any float
typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any_t;

constexpr int kDepth = 64;    // inputs of a tile
constexpr int kWaves = 4;     // along N

// grid (tiles of y, parts of K); part [parts, M, N] (gridDim.y > 1); depth: inputs of a part
// PER_CU: workgroups that share a CU
template <int TM, int TN, int STAGES, int PER_CU>
__global__ __launch_bounds__(64 * kWaves, PER_CU) void gemm_panel_q_kernel(
    __hip_bfloat16* __restrict__ y,         // [M, N]
    float* __restrict__ part,
    const __hip_bfloat16* __restrict__ x,   // [M, K]
    const unsigned char* __restrict__ w,    // int8 [N, K]
    const float* __restrict__ scale,        // [N]
    const int M, const int N, const int K, const int depth) {
  constexpr int BM = TM * 16, BN = TN * 16 * kWaves;
  constexpr int X_BYTES = BM * kDepth * 2, W_BYTES = BN * kDepth, STAGE = X_BYTES + W_BYTES;
  constexpr int X_LOADS = BM / 8, W_LOADS = BN / 16;   // 1 KB each: 8 rows of x, 16 of W
  constexpr int X_PASS = (X_LOADS + kWaves - 1) / kWaves, W_PASS = W_LOADS / kWaves;
  constexpr int LOADS = X_PASS + W_PASS;
  constexpr int AHEAD = 3;                // fragments of x on their way
  static_assert(TM >= TN && 2 * TM > AHEAD && STAGES >= 3, "what a tile's products hide");
  static_assert(STAGES * STAGE * PER_CU <= 160 * 1024, "LDS of a CU");
  __shared__ __align__(16) char lds[STAGES * STAGE];

  // neighbours in a run of blocks that one XCD gets share their columns of W
  const int m_tiles = (M + BM - 1) / BM, blocks = m_tiles * (N / BN);
  const int per_xcd = (blocks + 7) / 8, slot = blockIdx.x / 8;
  const int id = (blockIdx.x % 8) * per_xcd + slot;
  if (slot >= per_xcd || id >= blocks) return;
  const int k0 = blockIdx.y * depth;
  const int m0 = id % m_tiles * BM, n0 = id / m_tiles * BN;
  const int tiles = min(depth, K - k0) / kDepth;
  const int start = id / m_tiles % tiles;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, quad = lane >> 4;

  // (where there are fewer loads than waves some are made twice: all waves wait alike; rows
  // of a panel are found by 32 bits, see gemm_panel_plan)
  unsigned x_off[X_PASS], w_off[W_PASS];
#pragma unroll
  for (int p = 0; p < X_PASS; ++p) {
    const int r = (p * kWaves + wave) % X_LOADS * 8 + lane / 8;
    x_off[p] = (unsigned)min(r, M - 1 - m0) * (K * 2u) + ((lane % 8) ^ (r / 2 % 8)) * 16;
  }
#pragma unroll
  for (int p = 0; p < W_PASS; ++p) {
    const int r = (p * kWaves + wave) * 16 + lane / 4;
    w_off[p] = (unsigned)r * K + ((lane % 4) ^ (r / 4 % 4)) * 16;
  }
  const auto x_from = block_gemm::resource(x + (long)m0 * K + k0);
  const auto w_from = block_gemm::resource(w + (long)n0 * K + k0);
  // load p of a tile (past the last tile it is the last one again)
  auto load = [&](int buf, int tile, int p) {
    char* to = lds + buf * STAGE;
    tile = min(tile, tiles - 1) + start;
    if (tile >= tiles) tile -= tiles;
    if (p < X_PASS)
      block_gemm::load_lds(to + (p * kWaves + wave) % X_LOADS * 1024, x_from, x_off[p],
                           tile * (kDepth * 2));
    else
      block_gemm::load_lds(to + X_BYTES + ((p - X_PASS) * kWaves + wave) * 1024, w_from,
                           w_off[p - X_PASS], tile * kDepth);
  };

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_t{};

  // A lane's 16 weights of a column (chunk quad of its row) are its inputs of two matrix steps,
  // and x is read to match.
  auto x_frag = [&](const char* at, int s, int i) {
    const int r = i * 16 + col;
    return *reinterpret_cast<const bf16x8_t*>(at + r * (kDepth * 2) +
                                              ((quad * 2 + s) ^ (r / 2 % 8)) * 16);
  };
  auto w_chunk = [&](const char* at, int j) {
    const int r = (wave * TN + j) * 16 + col;
    return *reinterpret_cast<const u32x4_t*>(at + X_BYTES + r * kDepth + (quad ^ (r / 4 % 4)) * 16);
  };
  auto unpack = [&](const u32x4_t& c, int s) {
    union { unsigned u[4]; bf16x8_t v; } o;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const unsigned four = c[2 * s + d / 2] >> (d % 2 * 16);
      const float a = (float)(signed char)(four & 0xff);
      const float b = (float)(signed char)((four >> 8) & 0xff);
      // whole numbers of 8 bits: the upper half of the float is all of it
      o.u[d] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
    }
    return o.v;
  };

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
#pragma unroll
    for (int p = 0; p < LOADS; ++p) load(s, s, p);
  block_gemm::wait_loads<(STAGES - 2) * LOADS>();
  block_gemm::meet();
  u32x4_t c[TN];
  bf16x8_t wf[2][TN], xf[AHEAD];
#pragma unroll
  for (int j = 0; j < TN; ++j) c[j] = w_chunk(lds, j);
#pragma unroll
  for (int j = 0; j < TN; ++j) wf[0][j] = unpack(c[j], 0);
#pragma unroll
  for (int q = 0; q < AHEAD; ++q) xf[q] = x_frag(lds, q / TM, q % TM);

  int buf = 0;
  for (int t = 0; t < tiles; ++t) {
    const int after = buf + 1 == STAGES ? 0 : buf + 1, before = buf == 0 ? STAGES - 1 : buf - 1;
    const char* here = lds + buf * STAGE;
    const char* there = lds + after * STAGE;
    bf16x8_t xr[2 * TM + AHEAD];
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) xr[q] = xf[q];
#pragma unroll
    for (int q = 0; q < 2 * TM; ++q) {   // 16 rows of x and 32 inputs at a time
      const int s = q / TM, i = q % TM;
      if (q == TM) {
        // the next tile is here, and all have read the one before this one
        block_gemm::wait_loads<(STAGES - 3) * LOADS>();
        block_gemm::meet();
#pragma unroll
        for (int j = 0; j < TN; ++j) c[j] = w_chunk(there, j);
      }
#pragma unroll
      for (int p = 0; p < LOADS; ++p)
        if (s == 1 && p * TM / LOADS == i) load(before, t + STAGES - 1, p);
      const int f = q + AHEAD;
      xr[f] = f < 2 * TM ? x_frag(here, f / TM, f % TM)
                         : x_frag(there, (f - 2 * TM) / TM, (f - 2 * TM) % TM);
      // the weights of the next step, a column at a time
      if (s == 0 && i < TN) wf[1][i] = unpack(c[i], 1);
      if (s == 1 && i >= TM - TN) wf[0][i - (TM - TN)] = unpack(c[i - (TM - TN)], 0);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] =
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s][j], xr[q], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) xf[q] = xr[2 * TM + q];
    buf = after;
  }
  block_gemm::wait_loads<0>();   // LDS is not given back ahead of them

  const bool cut = gridDim.y > 1;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + (wave * TN + j) * 16 + quad * 4;
    const f32x4_t s = *reinterpret_cast<const f32x4_any_t*>(scale + n);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + i * 16 + col;
      if (m >= M) continue;
      f32x4_t v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = acc[i][j][r] * s[r];
      if (cut) {
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
