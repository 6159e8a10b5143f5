// The main loop of the large-tile products: C[BM, BN] += A[BM, K] B[BN, K]^T in bf16 on
// v_mfma_f32_16x16x32_bf16, both operands staged HBM -> LDS without registers
// (buffer_load ... lds, 16 bytes a lane), STAGES tiles of 64 inputs deep.
//
// LDS holds rows of 64 inputs (128 bytes, eight 16-byte chunks); chunk c of row r lies at
// chunk c ^ (r / 2 % 8), so that the 16 rows a fragment read touches cover all 64 banks.
// The write side is linear in the lane, so the swizzle is applied to what a lane fetches.
//
// One barrier a tile: wait for the own loads of this tile, meet, ask for the tile
// STAGES - 1 ahead (its buffer was read before the barrier), multiply: 16 rows of A at a
// time, read two ahead, the second half of B during the first.
//
// LDS traffic takes about as long as the products (256 x 256: 2048 cycles each a tile).
// Measured alone, bf16 N(K) x M, us: 28672 (4096) x 8192 1908 with global loads and the
// compiler's order, 1778 as here; 4096 (14336) x 8192 874, 799; 28672 (4096) x 512 111,
// 100.  A barrier before the last rows, so that the next tile's first reads hide behind
// them, 1790, 878, 110.
#pragma once

#include "common.h"

namespace block_gemm {

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int kDepth = 64;   // inputs of a tile

template <int N> DEVINLINE void wait_loads() {
  static_assert(N < 64, "vmcnt has six bits");
  // vmcnt(N), other counters left alone
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}

// vmcnt(N) and lgkmcnt(0)
template <int N> DEVINLINE void wait_loads_and_reads() {
  static_assert(N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0070);
}

// The waves meet; loads on their way to LDS stay on their way (a fence would wait for
// all of them).
DEVINLINE void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// 4 GB (or less) from a wave-uniform address on
DEVINLINE __amdgpu_buffer_rsrc_t resource(const void* from, unsigned size = 0xffffffff) {
  const unsigned long long at = reinterpret_cast<unsigned long long>(from);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)at);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(at >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void*>((unsigned long long)hi << 32 | lo), 0, size, 0x00027000);
}

// 16 (4) bytes a lane from `from` + offset (+ the uniform ahead) to lds + 16 (4) lane.
// Buffer loads: with a global one on its way the compiler has every read of LDS wait for
// all reads before it.
template <int HINT = 0>
DEVINLINE void load_lds(char* lds, __amdgpu_buffer_rsrc_t from, unsigned offset, int ahead) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      from, (__attribute__((address_space(3))) void*)lds, 16, offset, ahead, 0, HINT);
}
DEVINLINE void load_lds4(char* lds, __amdgpu_buffer_rsrc_t from, unsigned offset, int ahead) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      from, (__attribute__((address_space(3))) void*)lds, 4, offset, ahead, 0, 0);
}

template <int BM, int BN, int WM, int WN, int STAGES>
struct Block {
  static constexpr int kWaves = WM * WN;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int kTM = BM / WM / 16, kTN = BN / WN / 16;   // 16x16 tiles of a wave
  static constexpr int kAPass = BM / 8 / kWaves, kBPass = BN / 8 / kWaves;
  static constexpr int kStageBytes = (BM + BN) * kDepth * 2;
  static constexpr int kLds = STAGES * kStageBytes;
  static_assert(BM % (8 * kWaves) == 0 && BN % (8 * kWaves) == 0, "whole passes");
  static_assert(kLds <= 160 * 1024, "LDS of a CU");

  // a_row(r), b_row(r): byte offsets of row r of the block from a and b (32 bits)
  template <typename ARow, typename BRow>
  static DEVINLINE void run(f32x4_t (&acc)[kTM][kTN], char* lds, const char* a, const char* b,
                            const int K, ARow a_row, BRow b_row) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, quad = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;

    // this lane's rows and chunk of every pass: eight rows a wave and instruction
    unsigned a_off[kAPass], b_off[kBPass];
#pragma unroll
    for (int p = 0; p < kAPass; ++p) {
      const int r = (p * kWaves + wave) * 8 + lane / 8;
      a_off[p] = a_row(r) + ((lane % 8) ^ (r / 2 % 8)) * 16;
    }
#pragma unroll
    for (int p = 0; p < kBPass; ++p) {
      const int r = (p * kWaves + wave) * 8 + lane / 8;
      b_off[p] = b_row(r) + ((lane % 8) ^ (r / 2 % 8)) * 16;
    }
    const auto a_from = resource(a), b_from = resource(b);
    auto stage = [&](int buf, int tile) {
      char* to = lds + buf * kStageBytes + wave * 1024;
#pragma unroll
      for (int p = 0; p < kAPass; ++p)
        load_lds(to + p * kWaves * 1024, a_from, a_off[p], tile * (kDepth * 2));
#pragma unroll
      for (int p = 0; p < kBPass; ++p)
        load_lds(to + BM * kDepth * 2 + p * kWaves * 1024, b_from, b_off[p], tile * (kDepth * 2));
    };

    const int tiles = K / kDepth;
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
      if (s < tiles) stage(s, s);
    int buf = 0;
    for (int t = 0; t < tiles; ++t) {
      if (STAGES > 2 && t + 1 < tiles)
        wait_loads<(STAGES - 2) * (kAPass + kBPass)>();
      else
        wait_loads<0>();
      meet();
      if (t + STAGES - 1 < tiles) {
        int ahead = buf + STAGES - 1;
        if (ahead >= STAGES) ahead -= STAGES;
        stage(ahead, t + STAGES - 1);
      }
      const char* al = lds + buf * kStageBytes;
      const char* bl = al + BM * kDepth * 2;
      auto a_frag = [&](int q) {
        const int c = q / kTM * 4 + quad, r = (wm * kTM + q % kTM) * 16 + col;
        return *reinterpret_cast<const bf16x8_t*>(al + r * 128 + (c ^ (r / 2 % 8)) * 16);
      };
      auto b_frag = [&](int ks, int j) {
        const int c = ks * 4 + quad, r = (wn * kTN + j) * 16 + col;
        return *reinterpret_cast<const bf16x8_t*>(bl + r * 128 + (c ^ (r / 2 % 8)) * 16);
      };
      static_assert(kTN <= kTM, "the second half of B comes with the rows of the first of A");
      bf16x8_t bf[2][kTN], af[3];
#pragma unroll
      for (int j = 0; j < kTN; ++j) bf[0][j] = b_frag(0, j);
      af[0] = a_frag(0);
      af[1] = a_frag(1);
#pragma unroll
      for (int q = 0; q < 2 * kTM; ++q) {   // 16 rows of A and 32 inputs at a time
        if (q + 2 < 2 * kTM) af[(q + 2) % 3] = a_frag(q + 2);
        if (q < kTN) bf[1][q] = b_frag(1, q);
#pragma unroll
        for (int j = 0; j < kTN; ++j)
          acc[q % kTM][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[q % 3], bf[q / kTM][j],
                                                                    acc[q % kTM][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (++buf == STAGES) buf = 0;
    }
  }
};

}  // namespace block_gemm
