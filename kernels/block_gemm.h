// The main loop of the large-tile products: C[BM, BN] += A[BM, K] B[BN, K]^T in bf16 on
// v_mfma_f32_16x16x32_bf16, both operands staged HBM -> LDS without registers
// (global_load_lds, 16 bytes a lane), STAGES tiles of 64 inputs deep.
//
// LDS holds rows of 64 inputs (128 bytes, eight 16-byte chunks); chunk c of row r lies at
// chunk c ^ (r / 2 % 8), so that the 16 rows a fragment read touches cover all 64 banks.
// The write side is linear in the lane, so the swizzle is applied to what a lane fetches.
//
// One barrier a tile: wait for the own loads of this tile, meet, ask for the tile
// STAGES - 1 ahead (its buffer was read before the barrier), multiply.
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

// The waves meet; loads on their way to LDS stay on their way (a fence would wait for
// all of them).
DEVINLINE void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
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

  // a_row(r), b_row(r): byte offsets of row r of the block from a (anywhere) and b (32 bits)
  template <typename ARow, typename BRow>
  static DEVINLINE void run(f32x4_t (&acc)[kTM][kTN], char* lds, const char* a, const char* b,
                            const int K, ARow a_row, BRow b_row) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 15, quad = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;

    // this lane's rows and chunk of every pass: eight rows a wave and instruction
    unsigned long a_off[kAPass];
    unsigned b_off[kBPass];
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
    auto stage = [&](int buf, int tile) {
      char* to = lds + buf * kStageBytes;
      const char* at = a + (long)tile * (kDepth * 2);
      const char* bt = b + (long)tile * (kDepth * 2);
#pragma unroll
      for (int p = 0; p < kAPass; ++p)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) unsigned*)(at + a_off[p]),
            (__attribute__((address_space(3))) unsigned*)(to + (p * kWaves + wave) * 1024), 16, 0,
            0);
#pragma unroll
      for (int p = 0; p < kBPass; ++p)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) unsigned*)(bt + b_off[p]),
            (__attribute__((address_space(3))) unsigned*)(to + BM * kDepth * 2 +
                                                          (p * kWaves + wave) * 1024),
            16, 0, 0);
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
#pragma unroll
      for (int ks = 0; ks < kDepth / 32; ++ks) {
        bf16x8_t af[kTM], bf[kTN];
        const int c = ks * 4 + quad;
#pragma unroll
        for (int i = 0; i < kTM; ++i) {
          const int r = (wm * kTM + i) * 16 + col;
          af[i] = *reinterpret_cast<const bf16x8_t*>(al + r * 128 + (c ^ (r / 2 % 8)) * 16);
        }
#pragma unroll
        for (int j = 0; j < kTN; ++j) {
          const int r = (wn * kTN + j) * 16 + col;
          bf[j] = *reinterpret_cast<const bf16x8_t*>(bl + r * 128 + (c ^ (r / 2 % 8)) * 16);
        }
#pragma unroll
        for (int i = 0; i < kTM; ++i)
#pragma unroll
          for (int j = 0; j < kTN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
      }
      if (++buf == STAGES) buf = 0;
    }
  }
};

}  // namespace block_gemm
