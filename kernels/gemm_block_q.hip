// Products of more than one row with rounded weights: y[m, n] = sum_k x[m, k] W[n, k],
// W in int8 (a scale per row) or in 4 bits (offset 8, a scale per row and 128 inputs).
//
// The weights used to be widened by tensor ops (for 4 bits: masks, shifts, casts, a stack,
// two products, all in f32 in memory) ahead of a library product: 1.0 ms of 1.3 ms a
// llama-3-8b layer at 301 rows.  Now
//  - up to some hundreds of rows the product widens a tile's weights itself, between LDS
//    and the matrix unit: W crosses memory once, at its own size (gemm_panel_q.h, but
//    for small matrices);
//  - above, one kernel writes the widened matrix (bf16(q scale), bound by its bytes) for
//    the library's product, which is then the larger part and the faster one.
//
// In the product weights are whole numbers and scales are applied to 32-bit sums, as in
// gemm_stream.hip: int8 by conversion to f32 of which the upper half is all; 4 bits (in tiles; panels
// have n - 8 itself) as the bf16 pattern of 8 + n/2, with -12 times the sum of x added by a constant operand and the
// scale doubled.  A lane's 16 bytes of W hold the inputs of two matrix steps in int8, of four
// in 4 bits, and x is read to match.  x and W reach LDS without registers; chunks of a row are
// turned by the row: x by r (256-byte rows) or r / 2 (128), W by r / 2 (128) or r / 4 (64).
//
// Measured: four llama-3-8b layers around attention, 301 rows, int8: 5101 -> 1064 us with tiles of
// up to 64 x 128 whose weights every 64 rows widened again, -> 739 us with panels, -> 692 with the
// gate in the panel and widening spread over its products.
// 4 bits, in the same four layers, 196 rows: 932 -> 662 us with panels and the gate in them, 841 rows
// (widened for the library before) 2018 -> 1789.
// Widening 28672 x 4096: 61 us (5.8 TB/s).

#include <cmath>

#include "gemm_panel_q.h"

namespace {

using block_gemm::bf16x8_t;
using block_gemm::f32x4_t;

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2_t;

// DEPTH: inputs of a tile (4 bits: 128, a group of one scale).
template <int QB, int DEPTH, int BM, int BN, int WM, int WN, int STAGES>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_block_q_kernel(
    __hip_bfloat16* __restrict__ y,         // [M, N]
    const __hip_bfloat16* __restrict__ x,   // [M, K]
    const unsigned char* __restrict__ w,    // int8 [N, K] | packed [N, K / 2]
    const float* __restrict__ scale,        // [N] | [N, K / 128]
    const int M, const int N, const int K) {
  static_assert(QB == 8 || DEPTH == 128, "a tile of 4-bit weights is a group");
  constexpr int WAVES = WM * WN;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int AL = DEPTH / 8;                  // lanes (16 bytes) of an x row in a tile
  constexpr int WB = DEPTH * QB / 8;             // bytes of a W row in a tile
  constexpr int WL = WB / 16;                    // lanes a W row
  constexpr int CHUNKS = WL / 4;                 // 16-byte chunks of a lane's W row
  constexpr int STEPS = 16 * 8 / QB / 8;         // matrix steps of a chunk
  constexpr int A_PASS = BM * AL / 64 / WAVES;
  constexpr int B_LOADS = BN * WL / 64;          // 1 KB each, shared out over the waves
  constexpr int B_PASS = (B_LOADS + WAVES - 1) / WAVES;
  constexpr int S_PASS = QB == 4 ? 1 : 0;        // scales: 64 columns a load
  constexpr int A_BYTES = BM * DEPTH * 2, B_BYTES = BN * WB;
  constexpr int STAGE = A_BYTES + B_BYTES + (QB == 4 ? BN * 4 : 0);
  static_assert(BM * AL % (64 * WAVES) == 0 && BN * WL % 64 == 0 && BN % 64 == 0, "whole loads");
  __shared__ __align__(16) char lds[STAGES * STAGE];

  // neighbours in a run of blocks that one XCD gets share their columns of W
  const int m_tiles = (M + BM - 1) / BM, blocks = m_tiles * (N / BN);
  const int per_xcd = (blocks + 7) / 8, slot = blockIdx.x / 8;
  const int id = (blockIdx.x % 8) * per_xcd + slot;
  if (slot >= per_xcd || id >= blocks) return;
  const int m0 = id % m_tiles * BM, n0 = id / m_tiles * BN;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, quad = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  // a chunk's place in its row is turned by the row: rows of 256, 128, 64 bytes
  auto swz = [](int lanes, int r) { return lanes == 16 ? r % 16 : lanes == 8 ? r / 2 % 8 : r / 4 % 4; };

  unsigned a_off[A_PASS], b_off[B_PASS], s_off = 0;
#pragma unroll
  for (int p = 0; p < A_PASS; ++p) {
    const int r = (p * WAVES + wave) * (64 / AL) + lane / AL;
    a_off[p] = (min(m0 + r, M - 1) - m0) * (K * 2) + ((lane % AL) ^ swz(AL, r)) * 16;
  }
  // (where there are fewer loads than waves some are made twice: all waves wait alike)
#pragma unroll
  for (int p = 0; p < B_PASS; ++p) {
    const int r = (p * WAVES + wave) % B_LOADS * (64 / WL) + lane / WL;
    b_off[p] = r * (K * QB / 8) + ((lane % WL) ^ swz(WL, r)) * 16;
  }
  if constexpr (QB == 4) s_off = (wave % (BN / 64) * 64 + lane) * (K / 128) * 4;
  const auto x_from = block_gemm::resource(x + (long)m0 * K);
  const auto w_from = block_gemm::resource(w + (long)n0 * (K * QB / 8));
  const auto s_from = block_gemm::resource(QB == 4 ? scale + (long)n0 * (K / 128) : scale);
  auto stage = [&](int buf, int tile) {
    char* to = lds + buf * STAGE;
#pragma unroll
    for (int p = 0; p < A_PASS; ++p)
      block_gemm::load_lds(to + (p * WAVES + wave) * 1024, x_from, a_off[p], tile * (DEPTH * 2));
#pragma unroll
    for (int p = 0; p < B_PASS; ++p)
      block_gemm::load_lds(to + A_BYTES + (p * WAVES + wave) % B_LOADS * 1024, w_from, b_off[p],
                           tile * WB);
    if constexpr (QB == 4)
      block_gemm::load_lds4(to + A_BYTES + B_BYTES + wave % (BN / 64) * 256, s_from, s_off,
                              tile * 4);
  };

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_t{};
  bf16x8_t off;
#pragma unroll
  for (int j = 0; j < 8; ++j) off[j] = (short)0xc140;   // -12

  const int tiles = K / DEPTH;
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < tiles) stage(s, s);
  int buf = 0;
  for (int t = 0; t < tiles; ++t) {
    if (STAGES > 2 && t + 1 < tiles)
      block_gemm::wait_loads<(STAGES - 2) * (A_PASS + B_PASS + S_PASS)>();
    else
      block_gemm::wait_loads<0>();
    block_gemm::meet();
    if (t + STAGES - 1 < tiles) {
      int ahead = buf + STAGES - 1;
      if (ahead >= STAGES) ahead -= STAGES;
      stage(ahead, t + STAGES - 1);
    }
    const char* al = lds + buf * STAGE;
    const char* bl = al + A_BYTES;
    f32x4_t part[QB == 4 ? TM : 1][QB == 4 ? TN : 1], base[QB == 4 ? TM : 1];
    if constexpr (QB == 4) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        base[i] = f32x4_t{};
#pragma unroll
        for (int j = 0; j < TN; ++j) part[i][j] = f32x4_t{};
      }
    }
#pragma unroll
    for (int h = 0; h < CHUNKS; ++h) {
      u32x4_t c[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int r = (wn * TN + j) * 16 + col;
        c[j] = *reinterpret_cast<const u32x4_t*>(bl + r * WB + ((h * 4 + quad) ^ swz(WL, r)) * 16);
      }
#pragma unroll
      for (int st = 0; st < STEPS; ++st) {
        bf16x8_t xf[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int r = (wm * TM + i) * 16 + col;
          xf[i] = *reinterpret_cast<const bf16x8_t*>(
              al + r * (DEPTH * 2) + (((h * 4 + quad) * STEPS + st) ^ swz(AL, r)) * 16);
          if constexpr (QB == 4)
            base[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[i], off, base[i], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          union { unsigned u[4]; bf16x8_t v; } wf;
          if constexpr (QB == 8) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
              const unsigned two = c[j][2 * st + d / 2] >> (d % 2 * 16);
              const float a = (float)(signed char)(two & 0xff);
              const float b = (float)(signed char)((two >> 8) & 0xff);
              wf.u[d] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
            }
          } else {
            // even and odd weights to bits 3..6 of every byte, then to pairs
            const unsigned even = (c[j][st] << 3) & 0x78787878u;
            const unsigned odd = (c[j][st] >> 1) & 0x78787878u;
            wf.u[0] = __builtin_amdgcn_perm(odd, even, 0x0c040c00) | 0x41004100u;
            wf.u[1] = __builtin_amdgcn_perm(odd, even, 0x0c050c01) | 0x41004100u;
            wf.u[2] = __builtin_amdgcn_perm(odd, even, 0x0c060c02) | 0x41004100u;
            wf.u[3] = __builtin_amdgcn_perm(odd, even, 0x0c070c03) | 0x41004100u;
          }
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            f32x4_t& to = QB == 4 ? part[QB == 4 ? i : 0][QB == 4 ? j : 0] : acc[i][j];
            to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[i], wf.v, to, 0, 0, 0);
          }
        }
      }
    }
    if constexpr (QB == 4) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const float s =
            2.f * reinterpret_cast<const float*>(bl + B_BYTES)[(wn * TN + j) * 16 + col];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[i][j][r] = __builtin_fmaf(s, part[i][j][r] + base[i][r], acc[i][j][r]);
      }
    }
    if (++buf == STAGES) buf = 0;
  }

#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + (wn * TN + j) * 16 + col;
    const float s = QB == 8 ? scale[n] : 1.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + (wm * TM + i) * 16 + quad * 4 + r;
        if (m < M) y[(long)m * N + n] = __float2bfloat16(QB == 8 ? acc[i][j][r] * s : acc[i][j][r]);
      }
  }
}

// out[n, k] = bf16(q scale), 16 weights a thread; bound by the bytes in and out.
template <int QB>
__global__ __launch_bounds__(256) void widen_weight_kernel(
    __hip_bfloat16* __restrict__ out, const unsigned char* __restrict__ w,
    const float* __restrict__ scale, const long total, const int K) {
  for (long i = ((long)blockIdx.x * 256 + threadIdx.x) * 16; i < total;
       i += (long)gridDim.x * 4096) {
    const float s = QB == 8 ? scale[i / K] : scale[i / 128];
    Vec16<__hip_bfloat16> o[2];
    if constexpr (QB == 8) {
      const u32x4_t q = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(w + i));
#pragma unroll
      for (int j = 0; j < 16; ++j)
        o[j / 8].data[j % 8] =
            __float2bfloat16((float)(signed char)((q[j / 4] >> (j % 4 * 8)) & 0xff) * s);
    } else {
      const u32x2_t q = __builtin_nontemporal_load(reinterpret_cast<const u32x2_t*>(w + i / 2));
#pragma unroll
      for (int j = 0; j < 16; ++j)
        o[j / 8].data[j % 8] =
            __float2bfloat16(((float)((q[j / 8] >> (j % 8 * 4)) & 15) - 8.f) * s);
    }
    store16(out + i, o[0]);
    store16(out + i + 8, o[1]);
  }
}

// Tiles for small matrices, which panels have nothing to share over (int8: 64x64, and 32x64 where
// fewer; 4 bits: 32x64).  us, tiles | panels, columns x inputs: int8 2048 x 2048, 100 rows 10.3 | 10.2,
// 256 rows 10.5 | 12.3; 3072 x 2048, 128 rows 10.5 | 12.0, 301 rows 12.6 | 12.8, 384 rows 15.5 | 13.2
template <int QB>
void launch_block(__hip_bfloat16* y, const __hip_bfloat16* x, const unsigned char* w,
                  const float* scale, int M, int N, int K, hipStream_t stream) {
#define GO(DEPTH, BM, BN, WM, WN, ST)                                                        \
  hipLaunchKernelGGL((gemm_block_q_kernel<QB, DEPTH, BM, BN, WM, WN, ST>),                   \
                     dim3(((M + BM - 1) / BM * (N / BN) + 7) / 8 * 8), dim3(WM * WN * 64), 0, \
                     stream, y, x, w, scale, M, N, K)
  if constexpr (QB == 4) {
    GO(128, 32, 64, 1, 4, 3);
  } else {
    if ((M + 63L) / 64 * (N / 128) >= 150) GO(128, 64, 64, 1, 4, 2);
    else GO(128, 32, 64, 1, 4, 3);
  }
#undef GO
}

// Panels (gemm_panel_q.h) and how their time adds up, us: what a tile of 64 inputs takes with
// one workgroup on a CU and with as many as share one.  Fitted to some 5000 times (ten matrices
// from 1024 x 4096 to 28672 x 4096, 70 to 2048 rows, K cut over one to eight workgroups; 7 % rms);
// what it chooses is 0.9 % off the fastest panel in the mean (over 420 sizes, weights from memory).
// Workgroups are dealt to XCDs of 32 CUs, so rounds are counted there: over the whole chip a few
// more workgroups than CUs look like a second round that no XCD need have, and the other way
// around (1.2 % in the mean; 1280 x 8192, 800 rows 45 | 32 us, 1536 x 4096, 560 rows 20.6 | 18.1).
struct Panel {
  int tm, tn, per_cu;
  float one, full;
};
constexpr Panel kPanels[] = {{5, 1, 2, .232f, .423f}, {5, 2, 2, .347f, .598f},
                             {6, 2, 2, .373f, .648f}, {8, 1, 2, .319f, .551f},
                             {8, 2, 2, .582f, .784f}, {8, 2, 1, .482f, .482f},
                             {10, 2, 1, .550f, .550f}, {10, 4, 1, .985f, .985f}};

// Panels for 4 bits, likewise, over 1800 times (eleven matrices, 65 to 1000 rows; 6 % rms; the choice
// is 0.5 % off the fastest in the mean): weights are a quarter of what x is in LDS, so that panels of
// few rows of x and many columns pay, and two workgroups a CU, whose products hide the scaling of
// each other's sums.  us, tiles of up to 64 x 128 before | panels: 28672 x 4096, 128 rows 53 | 46, 196
// 97 | 67, 301 125 | 82, 600 229 | 161; 4096 x 14336, 80 rows 51 | 23, 196 72 | 43, 301 102 | 51; 6144 x
// 4096, 196 rows 32 | 27, 420 49 | 36; 4096 x 4096, 80 rows 17.1 | 12.9, 301 31 | 23; 1024 x 4096, 65 rows
// 17 | 8.2.
constexpr Panel kPanels4[] = {
    {5, 1, 2, .259f, .515f}, {5, 2, 2, .426f, .693f}, {6, 2, 2, .451f, .725f},
    {8, 1, 2, .350f, .619f}, {8, 2, 2, .623f, .867f}, {5, 4, 2, .679f, 1.076f},
    {4, 2, 2, .371f, .628f}};

float panel4_us(const Panel& p, int M, int N, int K, int parts) {
  const int blocks = (M + p.tm * 16 - 1) / (p.tm * 16) * (N / (p.tn * 64));
  const int wgs = (blocks + 7) / 8 * parts;   // of an XCD
  const int tiles = (K / 128 + parts - 1) / parts * 2, round = 32 * p.per_cu, left = wgs % round;
  float us = 4.3f + wgs / round * (p.full * tiles);
  if (left > 0) us += (left > 32 ? p.full : p.one) * tiles;
  if (parts > 1) us += 1.8f + 1.65e-6f * parts * M * N;
  return us;
}

// 32 x 64 tiles of 4 bits while they are at most two a CU and K is short: us, tiles | panels, 768 x 768,
// 301 rows 4.9 | 6.6; 4096 x 1024, 65 rows 6.0 | 8.3, 160 7.7 | 8.0, 301 (640 tiles) 10.1 | 8.4; 2048 x
// 2048, 65 rows 9.1 | 8.1, 224 9.5 | 11.4, 384 12.5 | 12.4; 512 x 2048, 301 rows 9.3 | 8.4, 700 9.5 | 10.7
float tiles4_us(int M, int N, int K) {
  const int all = ((M + 31) / 32 * (N / 64) + 7) / 8;   // of an XCD
  if (K > 2048 || all > 64) return 1e30f;
  return all <= 32 ? 2.4f + K / 128 * 0.44f : 2.6f + K / 128 * 0.62f;
}

float panel_us(const Panel& p, int M, int N, int K, int parts) {
  const int blocks = (M + p.tm * 16 - 1) / (p.tm * 16) * (N / (p.tn * 64));
  const int wgs = (blocks + 7) / 8 * parts;   // of an XCD
  const int tiles = (K / 64 + parts - 1) / parts, round = 32 * p.per_cu, left = wgs % round;
  float us = 2.6f + wgs / round * (p.full * tiles + 3.4f);
  if (left > 0) us += (left > 32 ? p.full : p.one) * tiles + 3.4f;
  if (parts > 1) us += 2.1f + 1.6e-6f * parts * M * N;   // their merge
  return us;
}

// Small matrices of short K stay with the tiles of launch_block while those are at most one to a CU,
// or three to nearly every one (as many as fit): there is nothing to share that a panel would save.
// us, tiles | panels: 768 x 768, 430 rows 5.5 | 6.6, 1000 rows 6.6 | 6.9; 128 x 512, 1000 rows
// 4.6 | 5.5; 3072 x 768, 1000 rows (768 tiles) 10.8 | 12.7.  Past one to a CU panels are up to 25 %
// faster (2048 x 1024, 640 rows, 320 tiles 9.7 | 8.0), and with few tiles of longer K, which
// panels cut, 10 % (128 x 2048).  (Below 256 inputs and past 320 rows panels are taken as before.)
bool small_tiles(int M, int N, int K) {
  if (K > 2048 || (long)N * K > 1 << 23) return false;
  if (M <= 320) return true;
  const long tiles = (M + 63L) / 64 * (N / 64);
  if (tiles > 736 && tiles <= 768) return K >= 256 && K <= 1024;
  return K >= 256 && tiles <= 256 && (K <= 1536 || tiles > 64);
}

}  // namespace

namespace {

// Panels for up to 64 rows, all of them in one: columns in K parts that fill the chip, as the
// streaming kernels' (gemm_stream.hip), but x is read by four times as many columns at a time, loads
// need no registers and weights no turn through LDS and back.  us, streaming | panels, int8: 28672 x
// 4096, 9 rows 27.6 | 24.5, 24 27.1 | 25.5, 40 36.8 | 27.4, 64 42.6 | 30.1; 4096 x 14336, 24 rows 17.4 |
// 16.6, 64 28.9 | 22.7; 6144 x 4096, 64 rows 18.9 | 14.8; 4096 x 4096, 40 rows 12.4 | 9.8; 2048 x 8192, 24 rows
// 12.2 | 9.1.  4 bits: 28672 x 4096, 24 rows 32.1 | 26.4, 64 46.6 | 29.8; 4096 x 14336, 24 rows 20.4 | 17.1,
// 64 33.0 | 20.6; 2048 x 8192, 24 rows 13.6 | 9.8; 8192 x 28672, 8 rows 62 | 45.
// Their times, fitted as above (to sixteen matrices, 2 to 64 rows; 4.5 % rms; the choice is 0.3 % off the
// best in the mean): as few rows are near the bytes of W, those at least.  int8, 4 bits:
struct FewPanel {
  int tm, tn;
  float one[2], full[2];
};
constexpr FewPanel kFewPanels[] = {
    {2, 1, {.198f, .219f}, {.347f, .458f}}, {2, 2, {.297f, .347f}, {.619f, .597f}},
    {3, 1, {.198f, .239f}, {.411f, .492f}}, {3, 2, {.330f, .349f}, {.658f, .617f}},
    {4, 1, {.231f, .249f}, {.436f, .494f}}, {4, 2, {.376f, .382f}, {.644f, .646f}}};
constexpr int kFewAt = 16;   // their number in a plan

int few_plan(int M, int N, int K, int qbits, bool gated, float& least) {
  const int q = qbits == 4, group = q ? 128 : 64;
  const float read = (q ? 0.269f * 0.5e-6f : 0.158f * 1e-6f) * N * K;
  int plan = 0;
  least = 1e30f;
  for (int i = 0; i < (int)(sizeof(kFewPanels) / sizeof(kFewPanels[0])); ++i) {
    const FewPanel& p = kFewPanels[i];
    if (16 * p.tm < M || N % (p.tn * 64) != 0) continue;
    for (int parts = 1; parts <= (gated ? 1 : 8) && (parts == 1 || K / parts >= 512); ++parts) {
      const int depth = (K / group + parts - 1) / parts;
      if ((K / group + depth - 1) / depth != parts) continue;   // no part is empty
      const int wgs = (N / (p.tn * 64) + 7) / 8 * parts, left = wgs % 64;   // of an XCD
      const int tiles = depth * (group / 64);
      float work = wgs / 64 * p.full[q] * tiles;
      if (left > 0) work += (left > 32 ? p.full[q] : p.one[q]) * tiles;
      float us = 3.2f + sqrtf(sqrtf(work * work * work * work + read * read * read * read));
      if (parts > 1) us += 1.75f + (q ? 2.7e-6f : 2.5e-6f) * parts * M * N;
      if (us < least) {
        plan = (kFewAt + i + 1) << 8 | parts;
        least = us;
      }
    }
  }
  return plan;
}

// The same for 4 bits; a gated one (N of both halves) has whole K
int panel4_plan(int M, int N, int K, bool gated, float& least) {
  int plan = gated ? 0 : 1;
  least = gated ? 1e30f : tiles4_us(M, N, K);
  for (int i = 0; i < (int)(sizeof(kPanels4) / sizeof(kPanels4[0])); ++i) {
    const Panel& p = kPanels4[i];
    if (N % (p.tn * 64) != 0) continue;
    // a panel's rows of x and of W lie inside 4 GB
    if (32L * p.tm * K >= 1L << 32 || 32L * p.tn * K >= 1L << 32) continue;
    for (int parts = 1; parts <= (gated ? 1 : 8) && (parts == 1 || K / parts >= 512); ++parts) {
      const int depth = (K / 128 + parts - 1) / parts;
      if ((K / 128 + depth - 1) / depth != parts) continue;   // no part is empty
      const float us = panel4_us(p, M, N, K, parts);
      if (us < least) {
        plan = (i + 1) << 8 | parts;
        least = us;
      }
    }
  }
  return plan;
}

}  // namespace

// Which panel, and how many workgroups K is cut over (each leaves a part of the result in f32),
// of eight tiles of 64 inputs at least: (panel << 8 | parts), or 1 where tiles of
// gemm_block_q_kernel do (small_tiles).  A function of shapes.
int gemm_panel_plan(int M, int N, int K, int qbits) {
  if (qbits == 4) {
    float us;
    return panel4_plan(M, N, K, false, us);
  }
  if (small_tiles(M, N, K)) return 1;
  int plan = 0;
  float least = 0.f;
  for (int i = 0; i < (int)(sizeof(kPanels) / sizeof(kPanels[0])); ++i) {
    if (N % (kPanels[i].tn * 64) != 0) continue;
    // a panel's rows of x and of W lie inside 4 GB
    if (32L * kPanels[i].tm * K >= 1L << 32 || 64L * kPanels[i].tn * K >= 1L << 32) continue;
    for (int parts = 1; parts <= 8 && (parts == 1 || K / parts >= 512); ++parts) {
      const int depth = (K / 64 + parts - 1) / parts;
      if ((K / 64 + depth - 1) / depth != parts) continue;   // no part is empty
      const float us = panel_us(kPanels[i], M, N, K, parts);
      if (plan == 0 || us < least) {
        plan = (i + 1) << 8 | parts;
        least = us;
      }
    }
  }
  return plan;
}

// The plan of a product of up to 64 rows by a panel, 0: the streaming kernels, which are as fast or
// faster for small matrices of short K and, in int8, up to 11 rows (us, streaming | panels: 33 rows,
// int8 4096 x 1024 6.2 | 7.2, 2048 x 2048 7.5 | 7.2, 8192 x 1024 9.3 | 6.5; 17 rows 4 bits 4096 x 4096
// 8.3 | 9.4, 16384 x 2048 13.1 | 10.5; 9 rows 6144 x 4096 9.8 | 10.4, 4 bits 10.4 |
// 11.3; 4 bits 2048 x 8192, 2 rows 9.9 | 9.1, 3584 x 8192 12.8 | 14.0, int8 2048 x 8192 8.3 | 8.5; int8 57344 x 8192, 8 rows 82 | 90, 14 rows
// 101 | 93, 8192 x 28672, 2 rows 52 | 46).
// A panel takes as long for 2 rows as for 32, the streaming kernels for 16 (and for 32, nearly):
//  - int8, 17 to 27 rows are as fast there but where W is so small that waves work alone in them (2^24: 1280 x 8192
//    0.75 of it, 512 x 14336 0.64; 1536 x 14336 11.2 | 12.2, 57344 x 7168 76 | 91, 6144 x 14336 22.3 | 24.3, but 4096 x
//    14336 1.00 to 0.97), shorter K up to 23 rows; from 28 on not where W is largest (57344 x 7168 86 | 93) or K is
//    longest and columns few (768 x 28672 17.2 | 18.2);
//  - up to 8 rows, many columns of long K: 4 bits 28672 x 8192 47 | 54, 16384 x 8192 27.7 | 31.0, but 16384 x 28672
//    80 | 83, 8 rows 0.86 of it; int8 14336 x 28672 77 | 89.
// Over 4698 products of 2 to 64 rows, 17 widths and 13 K, one is 3 % slower than streaming, the mean is 0.90 of it.
int gemm_panel_few_plan(int M, int N, int K, int qbits) {
  const long size = (long)N * K;
  bool takes;
  if (M < 2 || M > 64) takes = false;
  else if (M > 32) takes = K >= 2048 || size >= 8000000;
  else if (qbits == 4 && M > 16) takes = K >= 8192 || size >= 20000000;
  else if (qbits == 4)
    takes = (K >= 8192 && (N <= 2048 || (size >= 50000000 && (M > 8 || N <= 12288 || K >= 16384)))) ||
            (M > 8 && size >= 100000000);
  else if (M > 16)
    takes = (K >= 7168 && size <= 1 << 24) || (K >= 8192 && N >= 3584 && N <= 5120) ||
            (M > 23 && K >= 4096 && K < 8192 && size >= 20000000 && size < 200000000 &&
             (M > 27 || N < 14336)) ||
            (M > 27 && K >= 8192 && (K < 16384 || N > 2048));
  else
    takes = (K >= 16384 && (M > 6 || size <= 300000000)) ||
            (M > (K >= 5120 ? 11 : 13) && size >= 50000000);
  float us;
  return takes ? few_plan(M, N, K, qbits, false, us) : 0;
}

void launch_gemm_merge(__hip_bfloat16* y, const float* part, long plane, int parts, bool gated,
                       hipStream_t stream);

namespace {

// Without GATED: N columns of y; with it N / 2, of a plan for N with whole K
template <int QB, bool GATED>
void launch_panel(__hip_bfloat16* y, float* part, const __hip_bfloat16* x, const unsigned char* w,
                  const float* scale, int M, int N, int K, int plan, hipStream_t stream) {
  constexpr int kGroup = QB == 4 ? 128 : 64;
  const int parts = plan & 255, panel = (plan >> 8) - 1;
  const int depth = (K / kGroup + parts - 1) / parts * kGroup;
#define GO(I, TM, TN, STAGES, PER_CU)                                                         \
  case I: {                                                                                   \
    const int blocks = (M + TM * 16 - 1) / (TM * 16) * (N / (TN * 64));                       \
    hipLaunchKernelGGL((gemm_panel::gemm_panel_q_kernel<QB, TM, TN, STAGES, PER_CU, GATED>),  \
                       dim3((blocks + 7) / 8 * 8, parts), dim3(64 * gemm_panel::kWaves), 0,   \
                       stream, y, part, x, w, scale, M, GATED ? N / 2 : N, K, depth);         \
    break;                                                                                    \
  }
#define BOTH(I, ST4, ST8)                                                                     \
  GO(I, kPanelOf(I).tm, kPanelOf(I).tn, (QB == 4 ? ST4 : ST8), kPanelOf(I).per_cu)
#define FEW(I, ST4, ST8)                                                                      \
  GO(kFewAt + I, kFewPanels[I].tm, kFewPanels[I].tn, (QB == 4 ? ST4 : ST8), 2)
  constexpr auto kPanelOf = [](int i) constexpr { return QB == 4 ? kPanels4[i] : kPanels[i]; };
  switch (panel) {
    BOTH(0, 5, 5) BOTH(1, 5, 4) BOTH(2, 4, 4) BOTH(3, 4, 4) BOTH(4, 3, 3) BOTH(5, 4, 5) BOTH(6, 6, 4)
    FEW(0, 8, 8) FEW(1, 6, 6) FEW(2, 6, 6) FEW(3, 5, 5) FEW(4, 6, 6) FEW(5, 6, 4)
    default:
      if constexpr (QB == 8)
        switch (panel) {
          BOTH(7, 4, 4)
        }
  }
#undef FEW
#undef BOTH
#undef GO
  if (parts > 1) launch_gemm_merge(y, part, (long)M * N, parts, false, stream);
}

}  // namespace

// M >= 1, N % 128 == 0, K % 128 == 0; plan of gemm_panel_plan or gemm_panel_few_plan, its parts
// [parts, M, N]
void launch_gemm_block_q(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                         const unsigned char* w, const float* scale, int qbits, int M, int N,
                         int K, int plan, hipStream_t stream) {
  if (plan > 1 && qbits == 4)
    launch_panel<4, false>(y, part, x, w, scale, M, N, K, plan, stream);
  else if (plan > 1)
    launch_panel<8, false>(y, part, x, w, scale, M, N, K, plan, stream);
  else if (qbits == 4)
    launch_block<4>(y, x, w, scale, M, N, K, stream);
  else
    launch_block<8>(y, x, w, scale, M, N, K, stream);
}

// The plan of a gated product of M > 1 rows with [2 N, K], or 0 where the plain one and a launch for
// the gate (2.5 us, 4 bytes read and 2 written an output) are faster.  int8 past 64 rows: where the
// plain one's plan cuts K, as the gate is not in the panel then; others: the best panel with whole K
// against those two.  Up to 64 rows only for matrices that panels take as fast as the streaming kernels
// do (us, streaming and gate | gated panel, captured, int8: 28672 x 4096, 8 rows 27.9 | 26.4, 32 rows
// 31.2 | 27.9, 64 46.5 | 31.6; 16384 x 2048, 8 rows 11.7 | 9.9, 32 13.1 | 10.1; 4096 x 1024, 8 rows 5.9 | 6.1, 33
// rows 8.7 | 6.9; 4 bits 28672 x 4096, 2 rows 26.8 | 27.6, 4 rows 27.1 | 26.5, 16 rows 34.0 | 26.3).
// Few rows leave the gate little to save: not int8 up to 9 rows of long K, of few columns, or of large W (2 N x
// K: 57344 x 5120 53 | 71, 28672 x 7168 39 | 46, 10240 x 3584 12.6 | 14.0), nor 17 to 31 of the largest (57344 x 5120, 17
// rows 63 | 74), nor 4 bits of few columns, which all of K leaves CUs without (10240 x 3584, 10 rows 13.7 | 15.8, 14336 x
// 4096, 4 rows 16.4 | 18.1, 10 rows 18.3 | 18.2).  Of 4140 gated products nine are 3 % slower than streaming and
// gate (57344 x 1536, 2 rows, by 10, others by 5 at most), the mean is 0.89.
int gemm_panel_gated_plan(int M, int N, int K, int qbits) {
  if (M < 2 || N % 128 != 0 || K % 128 != 0 || (long)(N + 128) * K >= 1L << 32) return 0;
  float us, plain;
  int plan;
  if (M <= 64) {
    const long size = 2L * N * K;
    if (size < 24000000 && (K > 1024 || M <= 32)) return 0;
    if (qbits == 4
            ? M < 4 || (K >= 3584 && 2 * N <= 16384 && M < (2 * N <= 12288 ? 17 : 10))
            : (M < 10 && (size > 120000000 || K > 4096 || 2 * N < 14336)) ||
                  (M < 24 && (M < 12 || M > 16) && size >= 140000000) ||
                  (M > 16 && M < 32 && K >= 5120 && size >= 200000000))
      return 0;
    plan = few_plan(M, 2 * N, K, qbits, true, us);
    few_plan(M, 2 * N, K, qbits, false, plain);
  } else if (qbits == 4) {
    plan = panel4_plan(M, 2 * N, K, true, us);
    panel4_plan(M, 2 * N, K, false, plain);
  } else {
    plan = gemm_panel_plan(M, 2 * N, K, 8);
    return plan > 1 && (plan & 255) == 1 ? plan : 0;
  }
  return us < plain + 2.5f + 1.2e-6f * M * N ? plan : 0;
}

// y [M, N] = silu(x Wg^T) * (x Wu^T), W = [Wg; Wu] rounded, plan of gemm_panel_gated_plan
void launch_gemm_panel_gated(__hip_bfloat16* y, const __hip_bfloat16* x, const unsigned char* w,
                             const float* scale, int qbits, int M, int N, int K, int plan,
                             hipStream_t stream) {
  if (qbits == 4)
    launch_panel<4, true>(y, nullptr, x, w, scale, M, 2 * N, K, plan, stream);
  else
    launch_panel<8, true>(y, nullptr, x, w, scale, M, 2 * N, K, plan, stream);
}

// total = N * K, K % 128 == 0
void launch_widen_weight(__hip_bfloat16* out, const unsigned char* w, const float* scale,
                         int qbits, long total, int K, hipStream_t stream) {
  const long blocks = (total / 16 + 255) / 256;
  const dim3 grid(blocks < 16384 ? blocks : 16384);
  if (qbits == 8)
    hipLaunchKernelGGL(widen_weight_kernel<8>, grid, dim3(256), 0, stream, out, w, scale, total, K);
  else
    hipLaunchKernelGGL(widen_weight_kernel<4>, grid, dim3(256), 0, stream, out, w, scale, total, K);
}
