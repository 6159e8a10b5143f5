// The main loop of the products with many rows: C[BM, BN] += A[BM, K] B[BN, K]^T in bf16 on
// v_mfma_f32_16x16x32_bf16, one wave a SIMD, 256 x 256 by four waves.
//
// Bound by the matrix unit and, before it, by the chip's power: the clock falls to 1.7 GHz
// under it.  What counts is to keep the unit busy with as few bytes moved as possible:
//  - four waves of 128 x 128 read 128 KB of LDS a tile of 64 inputs, eight of 128 x 64 192 KB;
//    the sums fill all accumulation registers.
//  - Rows of 64 inputs, whole cache lines: with 32 (half lines; as much in flight, half of
//    the registers' turnover) every byte is asked for in two requests and the same loop
//    ran at 1.25 PFLOP/s instead of 1.5.
//  - Memory comes in slots of half of the rows of A and of B, SLOTS of them in LDS, each
//    asked for SLOTS - 1 half tiles ahead.  A half tile is half of the rows of A times all
//    of B, one half after the other; B's halves take turns in order from tile to tile
//    (A0 B0, A0 B1, A1 B1, A1 B0 | A0 B1, A0 B0, A1 B0, A1 B1), so that each quarter of the
//    products reads one half of an operand into the registers of one that is done with.
//  - One barrier a half tile.  Reads and loads stand between the products in source order.
// The accumulation registers are named in the products themselves (multiply below).
// Measured alone, us, the library | eight waves, two whole tiles in LDS | here, 4 slots (5):
//   rows x N (K): 8192 x 28672 (4096) 1412 | 1483 | 1325 (1351); 8192 x 4096 (14336) 609 |
//   722 | 618 (645); 8192 x 6144 (4096) 268 | 313 | 274 (286); 2949 x 28672 (4096) 531 | 600
//   | 527 (549); 512 x 28672 (4096) 91 | 115 | 96 (101).
#pragma once

#include "block_gemm.h"

namespace ring_gemm {

using block_gemm::bf16x8_t;
using block_gemm::f32x4_t;

constexpr int kDepth = 64;   // inputs of a tile

// HINT: of the loads of B (2: not to be kept in the caches)
template <int BM, int BN, int WM, int WN, int SLOTS, int HINT = 0>
struct Ring {
  static constexpr int kWaves = WM * WN;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int kTM = BM / WM / 16, kTN = BN / WN / 16;   // 16x16 tiles of a wave
  static constexpr int kHM = kTM / 2, kHN = kTN / 2;             // of half of its rows
  static constexpr int kABytes = BM / 2 * kDepth * 2, kSlot = (BM + BN) / 2 * kDepth * 2;
  static constexpr int kAPass = BM / 16 / kWaves, kBPass = BN / 16 / kWaves;
  static constexpr int kLoads = kAPass + kBPass;                 // a wave's of a slot
  static constexpr int kLds = SLOTS * kSlot;
  static_assert(kTM % 2 == 0 && kTN % 2 == 0, "halves");
  static_assert(BM % (16 * kWaves) == 0 && BN % (16 * kWaves) == 0, "whole passes");
  static_assert(kLds <= 160 * 1024, "LDS of a CU");
  static_assert((SLOTS - 1) * kLoads < 64, "vmcnt has six bits");

  // A sum stays in its accumulation registers: all 256 are in use, and the compiler's own
  // choice copies some of them in every turn.  Written out, a product is no matrix instruction
  // to the compiler, which adds no wait states: a form is sound only if between the products
  // sums are neither copied nor spilled and fragments come from LDS alone, and if `settle` is
  // the first to follow the last product.  tests/test_ring_products.py looks for that in the
  // built code; a new form, or a new compiler, has to pass it.
  static DEVINLINE void multiply(f32x4_t& acc, const bf16x8_t& a, const bf16x8_t& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  }
  // 18 wait states at most lie between a product and what reads its sum without the matrix
  // unit.  They are taken in the loop, behind the last product of the last turn: on the way out
  // of it the compiler copies sums.  One block, since a branch of its own would be moved there too.
  static DEVINLINE void settle(int turn, int turns) {
    asm volatile("s_cmp_lt_i32 %0, %1\n\ts_cbranch_scc1 1f\n\ts_nop 15\n\ts_nop 7\n1:"
                 ::"s"(turn), "s"(turns) : "scc");
    __builtin_amdgcn_sched_barrier(0);
  }
  // (the compiler would spill some of 256 that it takes to be wanted elsewhere)
  static DEVINLINE void keep(f32x4_t (&acc)[kTM][kTN]) {
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
      for (int j = 0; j < kTN; ++j) asm volatile("" : "+a"(acc[i][j]));
  }

  static DEVINLINE void clear(f32x4_t (&acc)[kTM][kTN]) {
#pragma unroll
    for (int i = 0; i < kTM; ++i)
#pragma unroll
      for (int j = 0; j < kTN; ++j) acc[i][j] = f32x4_t{};
  }
  // For results in 16-byte stores: if B's row r is column out_col(r), a lane's eight sums of
  // two neighbouring tiles j are eight neighbours, from column j * 16 + lane / 16 * 8 on.
  static DEVINLINE int out_col(int r) {
    return r / 32 * 32 + r % 16 / 4 * 8 + r / 16 % 2 * 4 + r % 4;
  }

  // acc[i][j][r]: row i * 16 + lane % 16 of A, row j * 16 + lane / 16 * 4 + r of B
  template <typename ARow, typename BRow>
  static DEVINLINE void run(f32x4_t (&acc)[kTM][kTN], char* lds, const char* a, const char* b,
                            const int K, ARow a_row, BRow b_row) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;

    // Where this lane's loads come from: eight rows a wave and instruction.  A slot's rows
    // are half of every wave's.
    unsigned a_off[2][kAPass], b_off[2][kBPass];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int p = 0; p < kAPass; ++p) {
        const int r = (p * kWaves + wave) * 8 + lane / 8;
        a_off[h][p] = a_row(r / (kHM * 16) * (kTM * 16) + h * (kHM * 16) + r % (kHM * 16)) +
                      ((lane % 8) ^ (r / 2 % 8)) * 16;
      }
#pragma unroll
      for (int p = 0; p < kBPass; ++p) {
        const int r = (p * kWaves + wave) * 8 + lane / 8;
        b_off[h][p] = b_row(r / (kHN * 16) * (kTN * 16) + h * (kHN * 16) + r % (kHN * 16)) +
                      ((lane % 8) ^ (r / 2 % 8)) * 16;
      }
    }
    // past the last tile: loads of nothing, so that the counts stay what they are
    const int n = K / kDepth;
    auto size = [&](int tile) {
      return (unsigned)__builtin_amdgcn_readfirstlane(tile < n ? -1 : 0);
    };
    // load p of half ha of A and hb of B of a tile
    auto load = [&](int p, char* slot, int ha, int hb, int tile, unsigned bytes) {
      char* to = slot + wave * 1024;
      if (p < kAPass)
        block_gemm::load_lds(to + p * kWaves * 1024, block_gemm::resource(a, bytes),
                             a_off[ha][p < kAPass ? p : 0], tile * (kDepth * 2));
      else
        block_gemm::load_lds<HINT>(to + kABytes + (p - kAPass) * kWaves * 1024,
                             block_gemm::resource(b, bytes),
                             b_off[hb][p < kAPass ? 0 : p - kAPass], tile * (kDepth * 2));
    };
    const int sw = (col / 2 % 8), c0 = (quad ^ sw) * 16, c1 = ((4 + quad) ^ sw) * 16;
    const int a_at = (wm * kHM * 16 + col) * 128, b_at = kABytes + (wn * kHN * 16 + col) * 128;
    auto read_a = [&](bf16x8_t (&f)[2 * kHM], const char* slot, int q) {
      f[q] = *reinterpret_cast<const bf16x8_t*>(slot + a_at + (q < kHM ? c0 : c1) +
                                                q % kHM * 2048);
    };
    auto read_b = [&](bf16x8_t (&f)[2 * kHN], const char* slot, int q) {
      f[q] = *reinterpret_cast<const bf16x8_t*>(slot + b_at + (q < kHN ? c0 : c1) +
                                                q % kHN * 2048);
    };

    // The order of the halves, two tiles in a round: A0 B0, A1 B1 | A0 B1, A1 B0
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
#pragma unroll
      for (int p = 0; p < kLoads; ++p)
        load(p, lds + s * kSlot, s % 2, (s + 1) / 2 % 2, s / 2, size(s / 2));
    block_gemm::wait_loads<(SLOTS - 1) * kLoads>();
    block_gemm::meet();
    bf16x8_t fa0[2 * kHM], fa1[2 * kHM], fb0[2 * kHN], fb1[2 * kHN];
#pragma unroll
    for (int q = 0; q < 2 * kHM; ++q) read_a(fa0, lds, q);
#pragma unroll
    for (int q = 0; q < 2 * kHN; ++q) read_b(fb0, lds, q);

    int at = 0, next = 1;    // places of the slot that has been read and of the next one
    // A quarter of a tile's products, the reads of a half and half of the loads in between
    auto quarter = [&](int i0, int j0, bf16x8_t (&fa)[2 * kHM], bf16x8_t (&fb)[2 * kHN],
                       int reads, auto read, int first, int last, auto ask) {
      constexpr int kProducts = 2 * kHM * kHN;
#pragma unroll
      for (int q = 0; q < kProducts; ++q) {
        const int ks = q / (kHM * kHN), i = q / kHN % kHM, jj = q % kHN;
        const int j = i % 2 ? kHN - 1 - jj : jj;
#pragma unroll
        for (int r = 0; r < reads; ++r)   // in the first half of the products, if they fit
          if (r * (2 * reads > kProducts ? kProducts : kProducts / 2) / reads == q) read(r);
        const int each = kProducts / (last - first);
#pragma unroll
        for (int l = first; l < last; ++l)
          if (min((l - first) * kProducts / (last - first) + each / 2 + 1, kProducts - 1) == q)
            ask(l);
        multiply(acc[i0 + i][j0 + j], fb[ks * kHN + j], fa[ks * kHM + i]);
        if (q % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
    };
    // what begins a half of a tile: the slot before has been read by all, the next is there
    auto begin = [&] {
      block_gemm::wait_loads_and_reads<(SLOTS - 2) * kLoads>();
      block_gemm::meet();
    };
    auto advance = [&] {
      at = next;
      if (++next == SLOTS) next = 0;
    };
    for (int t = 0; t < n; t += 2) {   // (an odd last tile's neighbour is zero)
      {
        // even tile: A0 B0, A0 B1 (reading B1, A1), A1 B1, A1 B0 (reading A0', B1')
        constexpr int kAhead = SLOTS;
        begin();
        char* here = lds + at * kSlot;
        const char* there = lds + next * kSlot;
        int tile = t + kAhead / 2;
        unsigned bytes = size(tile);
        auto ask0 = [&](int p) { load(p, here, SLOTS % 2, (SLOTS + 1) / 2 % 2, tile, bytes); };
        quarter(0, 0, fa0, fb0, 2 * kHN, [&](int q) { read_b(fb1, there, q); }, 0, kLoads / 2,
                ask0);
        quarter(0, kHN, fa0, fb1, 2 * kHM, [&](int q) { read_a(fa1, there, q); }, kLoads / 2,
                kLoads, ask0);
        advance();
        begin();
        char* here1 = lds + at * kSlot;
        const char* there1 = lds + next * kSlot;
        int tile1 = t + (SLOTS + 1) / 2;
        unsigned bytes1 = size(tile1);
        auto ask1 = [&](int p) {
          load(p, here1, (SLOTS + 1) % 2, (SLOTS + 2) / 2 % 2, tile1, bytes1);
        };
        quarter(kHM, kHN, fa1, fb1, 2 * kHM, [&](int q) { read_a(fa0, there1, q); }, 0,
                kLoads / 2, ask1);
        quarter(kHM, 0, fa1, fb0, 2 * kHN, [&](int q) { read_b(fb1, there1, q); }, kLoads / 2,
                kLoads, ask1);
        advance();
      }
      {
        // odd tile: A0 B1, A0 B0 (reading B0, A1), A1 B0, A1 B1 (reading A0', B0')
        begin();
        char* here = lds + at * kSlot;
        const char* there = lds + next * kSlot;
        int tile = t + 1 + SLOTS / 2;
        unsigned bytes = size(tile);
        auto ask0 = [&](int p) { load(p, here, SLOTS % 2, (SLOTS + 3) / 2 % 2, tile, bytes); };
        quarter(0, kHN, fa0, fb1, 2 * kHN, [&](int q) { read_b(fb0, there, q); }, 0, kLoads / 2,
                ask0);
        quarter(0, 0, fa0, fb0, 2 * kHM, [&](int q) { read_a(fa1, there, q); }, kLoads / 2,
                kLoads, ask0);
        advance();
        begin();
        char* here1 = lds + at * kSlot;
        const char* there1 = lds + next * kSlot;
        int tile1 = t + 1 + (SLOTS + 1) / 2;
        unsigned bytes1 = size(tile1);
        auto ask1 = [&](int p) {
          load(p, here1, (SLOTS + 1) % 2, (SLOTS + 4) / 2 % 2, tile1, bytes1);
        };
        quarter(kHM, 0, fa1, fb0, 2 * kHM, [&](int q) { read_a(fa0, there1, q); }, 0, kLoads / 2,
                ask1);
        quarter(kHM, kHN, fa1, fb1, 2 * kHN, [&](int q) { read_b(fb0, there1, q); }, kLoads / 2,
                kLoads, ask1);
        __builtin_amdgcn_sched_barrier(0);
        settle(t + 2, n);
        advance();
      }
    }
    block_gemm::wait_loads<0>();
    keep(acc);
  }
};

}  // namespace ring_gemm
