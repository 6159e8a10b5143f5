// The first of an adapter's two products for the tokens of a mixed batch (lora_bgmv.hip), as a
// workgroup's work: by itself, or beside the workgroups of the product whose deltas these become
// (gemm_ring.hip).
#pragma once

#include "common.h"

namespace lora {

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int kShrinkWaves = 4;
constexpr int kWindow = 256;   // tokens that are grouped by adapter

struct Shrink {
  float* tmp;                     // [cuts, T, PR]
  const __hip_bfloat16* x;        // [T, K]
  const __hip_bfloat16* a_stack;  // [L, PR, K]
  const int* slots;               // [T]
  int T, PR, K, cuts;
};

constexpr int shrink_lds(int tiles) { return kShrinkWaves * (tiles * 1024 + 64); }

// Groups of a window of n tokens that L adapters leave at most.
__host__ __device__ inline int groups_of(int n, int L) { return n / 16 + (L < n ? L : n); }

// A workgroup (cut of K, group of 16 tokens): of the window of kWindow tokens from t0 on, those that
// have one adapter, in any order, from the `first`-th on; it ends at once where there are no more.
// ANY: the first-th group of all adapters' groups, `slot` is the number of adapters.  Tokens without
// an adapter are left unwritten.  TILES 16-wide tiles of PR from row `row0` on; lds:
// shrink_lds(TILES) bytes.
//
// Groups of neighbours instead read every adapter of a mixed batch's 16 tokens for one or
// two of them.  32 adapters of rank 8 dealt out at random, 1024 x 4096, us with expand, a
// token a workgroup, neighbours, windows: 256 tokens 10.3 17.4 9.5, 1000 14.4 33.9 15.1.
template <int TILES, bool ANY>
DEVINLINE void shrink(const Shrink& s, const int cut, int slot, const int t0, int first,
                      const int row0, char* lds) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, quad = lane >> 4;
  f32x4_t* all = reinterpret_cast<f32x4_t*>(lds);                        // [waves][TILES][64]
  int* group = reinterpret_cast<int*>(lds + kShrinkWaves * TILES * 1024) + wave * 16;
  int slot_of[kWindow / 64], found = 0;
#pragma unroll
  for (int i = 0; i < kWindow / 64; ++i)
    slot_of[i] = t0 + i * 64 + lane < s.T ? s.slots[t0 + i * 64 + lane] : -1;
  if constexpr (ANY) {
    const int adapters = slot;
    for (slot = 0; slot < adapters; ++slot) {
      int n = 15;
#pragma unroll
      for (int i = 0; i < kWindow / 64; ++i) n += __popcll(__ballot(slot_of[i] == slot));
      if (first < n / 16) break;
      first -= n / 16;
    }
    if (slot == adapters) return;
    first *= 16;
  }
#pragma unroll
  for (int i = 0; i < kWindow / 64; ++i) {
    const unsigned long long has = __ballot(slot_of[i] == slot);
    const int at = found + __popcll(has & ((1ull << lane) - 1)) - first;
    if (slot_of[i] == slot && at >= 0 && at < 16) group[at] = t0 + i * 64 + lane;
    found += __popcll(has);
  }
  const int tokens = min(found - first, 16);
  if (tokens <= 0) return;
  // other lanes of this wave read it: LDS keeps a wave's order, the compiler has to
  asm volatile("" ::: "memory");
  const int own = group[min(col, tokens - 1)];

  const __hip_bfloat16* xr = s.x + (long)own * s.K + quad * 8;
  const __hip_bfloat16* ar[TILES];
#pragma unroll
  for (int j = 0; j < TILES; ++j)
    ar[j] = s.a_stack + ((long)slot * s.PR + min(row0 + j * 16 + col, s.PR - 1)) * s.K + quad * 8;
  f32x4_t acc[TILES];
#pragma unroll
  for (int j = 0; j < TILES; ++j) acc[j] = f32x4_t{};

  const int steps = (s.K + 31) / 32, stride = s.cuts * kShrinkWaves;
  constexpr int AHEAD = TILES <= 4 ? 4 : 2;
  for (int s0 = cut * kShrinkWaves + wave; s0 < steps; s0 += AHEAD * stride) {
    bf16x8_t xf[AHEAD], af[AHEAD][TILES];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int k = (s0 + u * stride) * 32;
      const bool in = k + quad * 8 < s.K;   // K % 8 == 0: a lane's eight inputs are in or out
      xf[u] = in ? *reinterpret_cast<const bf16x8_t*>(xr + k) : bf16x8_t{};
#pragma unroll
      for (int j = 0; j < TILES; ++j)
        af[u][j] = in ? *reinterpret_cast<const bf16x8_t*>(ar[j] + k) : bf16x8_t{};
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
#pragma unroll
      for (int j = 0; j < TILES; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[u], af[u][j], acc[j], 0, 0, 0);
  }

#pragma unroll
  for (int j = 0; j < TILES; ++j) all[(wave * TILES + j) * 64 + lane] = acc[j];
  __syncthreads();
  for (int j = wave; j < TILES; j += kShrinkWaves) {
    f32x4_t v = all[j * 64 + lane];
#pragma unroll
    for (int w = 1; w < kShrinkWaves; ++w) v += all[(w * TILES + j) * 64 + lane];
    const int r = row0 + j * 16 + col;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = quad * 4 + i, t = __shfl(own, m, 64);
      if (m < tokens && r < s.PR) s.tmp[((long)cut * s.T + t) * s.PR + r] = v[i];
    }
  }
}

}  // namespace lora

int lora_shrink_cuts(int T, int K);
