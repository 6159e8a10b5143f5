// Batched multi-LoRA products.
//
// Mixed-adapter batches carry a per-token adapter slot (-1 = no adapter); weights of the
// active adapters are stacked host-side, for up to three projections of one input side
// by side (q, k, v; gate, up):
//   A_stack [L, P R, K]   (shrink:  tmp[t] = A[slot(t)] · x[t])
//   B_stack [L, V, R]     (expand:  out[t, col(v)] += scale_s · B[slot(t), v] · tmp[t, p(v)])
// with R padded to the largest rank (padded rows / columns are zero) and V the columns of
// the projections one after the other.
//
// bf16, shrink: 16 tokens of one adapter a workgroup (taken from a window of 256, see the
// kernel), K cut over workgroups and waves, both operands straight from L2 into
// v_mfma_f32_16x16x32_bf16.  The former kernel took a token a workgroup and a rank at a
// time, each with its own wave reduction.  expand: one column a thread, the tokens of a
// workgroup in turn, a row of B kept while the adapter stays the same, f32 sums in f32.
// Both are bound by launch and load latency at decode sizes; at prompt sizes expand by the
// read and write of out.
//
// Layers of 4096 wide rows, 61 tokens of 4 adapters of rank 16: 7 + 7 launches of 25 and
// 5 us were 4 + 4 of 4.6 and 4.0 to 7.8; of these the shrinks go beside their products now
// (gemm_ring_lora), a pass of 604 us is one of 548.  2048 tokens: shrink 23 us, expand into 4096 columns 14
// and into 28672 102 (by the matrix unit some 75), where reading and writing out takes 51.
//
// f32 and f16: one token per workgroup in both,
//   shrink: 4 waves split K; each (wave, r) pair accumulates a partial dot,
//           folded across lanes by shfl and across waves in LDS.  tmp is f32.
//   expand: R <= 64 fits a lane-resident tmp row; each thread owns one
//           output column and walks r with the B row loads coalesced.

#include "lora_shrink.h"
#include <float.h>

// ---------------------------------------------------------------------------
// shrink: tmp[T, R] (f32) = A[slot(t)] · x[t]
// grid (T), block 256
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void lora_shrink_kernel(
    float* __restrict__ tmp,        // [T, R]
    const T* __restrict__ x,        // [T, K]
    const T* __restrict__ a_stack,  // [L, R, K]
    const int* __restrict__ slots,  // [T]
    const int R,
    const int K) {
  const int t = blockIdx.x;
  const int slot = slots[t];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;

  if (slot < 0) {
    for (int r = threadIdx.x; r < R; r += blockDim.x) tmp[(long)t * R + r] = 0.f;
    return;
  }

  const T* x_row = x + (long)t * K;
  const T* a_base = a_stack + (long)slot * R * K;

  // waves split K into quarters (rounded to 16B so k_lo stays aligned)
  constexpr int EV = Vec16<T>::kElems;
  const int k_per_wave = ((K + 3) / 4 + EV - 1) / EV * EV;
  const int k_lo = min(wave * k_per_wave, K);
  const int k_hi = min(k_lo + k_per_wave, K);

  __shared__ float lds[4][64];  // [wave][r] partials (R <= 64)
  for (int r = 0; r < R; ++r) {
    float acc = 0.f;
    const T* a_row = a_base + (long)r * K;
    // lanes cover every aligned 16B chunk in [k_lo, k_hi) (K % 8 == 0
    // enforced by the binding)
    constexpr int E = Vec16<T>::kElems;
    for (int k = k_lo + lane * E; k + E <= k_hi; k += 64 * E) {
      const Vec16<T> xv = load16(x_row + k);
      const Vec16<T> av = load16(a_row + k);
#pragma unroll
      for (int j = 0; j < Vec16<T>::kElems; ++j)
        acc += ScalarOps<T>::to_f32(xv.data[j]) * ScalarOps<T>::to_f32(av.data[j]);
    }
    acc = wave_reduce_sum(acc);
    if (lane == 0) lds[wave][r] = acc;
  }
  __syncthreads();
  for (int r = threadIdx.x; r < R; r += blockDim.x)
    tmp[(long)t * R + r] = lds[0][r] + lds[1][r] + lds[2][r] + lds[3][r];
}

// ---------------------------------------------------------------------------
// expand: out[t, off + n] += scale[slot] * sum_r B[slot][n, r] * tmp[t, r]
// grid (T, ceil(N/256)), block 256
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void lora_expand_kernel(
    T* __restrict__ out,            // [T, out_w]
    const float* __restrict__ tmp,  // [T, R]
    const T* __restrict__ b_stack,  // [L, N, R]
    const int* __restrict__ slots,  // [T]
    const float* __restrict__ scales,  // [L]
    const int R,
    const int N,
    const int out_w,
    const int off) {
  const int t = blockIdx.x;
  const int slot = slots[t];
  if (slot < 0) return;
  const int n = blockIdx.y * 256 + threadIdx.x;
  if (n >= N) return;

  __shared__ float tmp_lds[64];
  if (threadIdx.x < R) tmp_lds[threadIdx.x] = tmp[(long)t * R + threadIdx.x];
  __syncthreads();

  const T* b_row = b_stack + ((long)slot * N + n) * R;
  float acc = 0.f;
  for (int r = 0; r < R; ++r)
    acc += ScalarOps<T>::to_f32(b_row[r]) * tmp_lds[r];

  T* o = out + (long)t * out_w + off + n;
  *o = ScalarOps<T>::from_f32(ScalarOps<T>::to_f32(*o) + acc * scales[slot]);
}

template <typename T>
void launch_lora_shrink(float* tmp, const T* x, const T* a_stack,
                        const int* slots, int Tn, int R, int K,
                        hipStream_t stream) {
  hipLaunchKernelGGL(lora_shrink_kernel<T>, dim3(Tn), dim3(256), 0, stream,
                     tmp, x, a_stack, slots, R, K);
}

template <typename T>
void launch_lora_expand(T* out, const float* tmp, const T* b_stack,
                        const int* slots, const float* scales, int Tn, int R,
                        int N, int out_w, int off, hipStream_t stream) {
  hipLaunchKernelGGL(lora_expand_kernel<T>, dim3(Tn, (N + 255) / 256),
                     dim3(256), 0, stream, out, tmp, b_stack, slots, scales, R,
                     N, out_w, off);
}

// ---------------------------------------------------------------------------
// bf16
// ---------------------------------------------------------------------------

// virtual column v of projection p (v < end[p]) is column v + shift[p] of out
struct LoraCols {
  int end[3], shift[3];
};

bool lora_tiles_win(int T, int L, int R, int W);

namespace {

using lora::kShrinkWaves;

// grid (cuts, adapters, windows x kWindow / 16 groups): groups are numbered slowest, so that the
// ones that have tokens lie next to each other and on all XCDs
template <int TILES>   // 16-wide tiles of PR
__global__ __launch_bounds__(64 * kShrinkWaves) void lora_shrink_tile_kernel(
    float* __restrict__ tmp, const __hip_bfloat16* __restrict__ x,
    const __hip_bfloat16* __restrict__ a_stack, const int* __restrict__ slots, const int T,
    const int PR, const int K) {
  __shared__ __align__(16) char lds[lora::shrink_lds(TILES)];
  constexpr int GROUPS = lora::kWindow / 16;
  lora::shrink<TILES, false>(lora::Shrink{tmp, x, a_stack, slots, T, PR, K, (int)gridDim.x},
                             blockIdx.x, blockIdx.y, blockIdx.z / GROUPS * lora::kWindow,
                             blockIdx.z % GROUPS * 16, 0, lds);
}

// The cuts' sums of a workgroup's tokens.  FEW: eight parts are asked for at once.
template <int R, int TOKENS, bool FEW>
DEVINLINE void add_cuts(float (&sums)[TOKENS][3 * R], const float* __restrict__ tmp, const int T,
                        const int t0, const int tokens, const int PR, const int cuts) {
  for (int i = threadIdx.x; i < tokens * PR; i += 256) {
    float s = 0.f;
    if constexpr (FEW) {
      for (int c0 = 0; c0 < cuts; c0 += 8) {
        float part[8];
#pragma unroll
        for (int c = 0; c < 8; ++c)
          part[c] = tmp[((long)min(c0 + c, cuts - 1) * T + t0) * PR + i];
#pragma unroll
        for (int c = 0; c < 8; ++c)
          if (c0 + c < cuts) s += part[c];
      }
    } else {
      for (int c = 0; c < cuts; ++c) s += tmp[((long)c * T + t0) * PR + i];
    }
    sums[i / PR][i % PR] = s;
  }
}

// grid (ceil(V / 256), ceil(T / TOKENS))
template <int R, int TOKENS>
__global__ __launch_bounds__(256) void lora_expand_tile_kernel(
    __hip_bfloat16* __restrict__ out,            // [T, out_w]
    const float* __restrict__ tmp,               // [cuts, T, PR]
    const __hip_bfloat16* __restrict__ b_stack,  // [L, V, R]
    const int* __restrict__ slots, const float* __restrict__ scales, const LoraCols cols,
    const int T, const int PR, const int V, const int out_w, const int cuts) {
  __shared__ float sums[TOKENS][3 * R];
  __shared__ int own[TOKENS];
  const int t0 = blockIdx.y * TOKENS, v = blockIdx.x * 256 + threadIdx.x;
  const int tokens = min(TOKENS, T - t0);
  if (threadIdx.x < TOKENS)
    own[threadIdx.x] = threadIdx.x < tokens ? slots[t0 + threadIdx.x] : -1;
  __syncthreads();
  for (int i = threadIdx.x; i < tokens * PR; i += 256) {
    const int t = i / PR;
    float s = 0.f;
    if (own[t] >= 0)
      for (int c = 0; c < cuts; ++c) s += tmp[((long)c * T + t0) * PR + i];
    sums[t][i % PR] = s;
  }
  __syncthreads();
  if (v >= V) return;
  const int p = v < cols.end[0] ? 0 : v < cols.end[1] ? 1 : 2;
  __hip_bfloat16* o = out + (long)t0 * out_w + v + cols.shift[p];
  float was[TOKENS];
#pragma unroll
  for (int t = 0; t < TOKENS; ++t)
    was[t] = t < tokens ? __bfloat162float(o[(long)t * out_w]) : 0.f;

  Vec16<__hip_bfloat16> b[R / 8];
  float scale = 0.f;
  int cur = -1;
#pragma unroll
  for (int t = 0; t < TOKENS; ++t) {
    const int slot = __builtin_amdgcn_readfirstlane(own[t]);
    if (slot < 0) continue;
    if (slot != cur) {
      cur = slot;
      scale = scales[slot];
#pragma unroll
      for (int j = 0; j < R / 8; ++j) b[j] = load16(b_stack + ((long)slot * V + v) * R + j * 8);
    }
    float acc = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r)
      acc = __builtin_fmaf(__bfloat162float(b[r / 8].data[r % 8]), sums[t][p * R + r], acc);
    o[(long)t * out_w] = __float2bfloat16(was[t] + acc * scale);
  }
}

// The same for few tokens, which are a chain of latencies: what was in out, the cuts' sums and,
// where they fit, the rows of B for all tokens are asked for at once (61 tokens, rank 16, 4096
// columns, K in 16 cuts: 4.5 -> 3.4 us).
template <int R>
__global__ __launch_bounds__(256) void lora_expand_few_kernel(
    __hip_bfloat16* __restrict__ out,            // [T, out_w]
    const float* __restrict__ tmp,               // [cuts, T, PR]
    const __hip_bfloat16* __restrict__ b_stack,  // [L, V, R]
    const int* __restrict__ slots, const float* __restrict__ scales, const LoraCols cols,
    const int T, const int PR, const int V, const int out_w, const int cuts) {
  constexpr int TOKENS = 2;
  constexpr bool AHEAD = TOKENS * R <= 64;
  __shared__ float sums[TOKENS][3 * R];
  const int t0 = blockIdx.y * TOKENS, v = blockIdx.x * 256 + threadIdx.x;
  const int tokens = min(TOKENS, T - t0);
  int own[TOKENS];
#pragma unroll
  for (int t = 0; t < TOKENS; ++t)
    own[t] = __builtin_amdgcn_readfirstlane(t < tokens ? slots[t0 + t] : -1);
  const int p = v < cols.end[0] ? 0 : v < cols.end[1] ? 1 : 2;
  __hip_bfloat16* o = out + (long)t0 * out_w + v + cols.shift[p];
  __hip_bfloat16 was[TOKENS];
  Vec16<__hip_bfloat16> b[AHEAD ? TOKENS : 1][R / 8];
  float scale[TOKENS];
#pragma unroll
  for (int t = 0; t < TOKENS; ++t) {
    if (own[t] < 0) continue;
    scale[t] = scales[own[t]];
    if (v >= V) continue;
    was[t] = o[(long)t * out_w];
    if constexpr (AHEAD) {
#pragma unroll
      for (int j = 0; j < R / 8; ++j) b[t][j] = load16(b_stack + ((long)own[t] * V + v) * R + j * 8);
    }
  }
  // (tokens without an adapter: whatever is there, which is not used)
  add_cuts<R, TOKENS, true>(sums, tmp, T, t0, tokens, PR, cuts);
  __syncthreads();
  if (v >= V) return;
  int cur = -1;
#pragma unroll
  for (int t = 0; t < TOKENS; ++t) {
    if (own[t] < 0) continue;
    if constexpr (!AHEAD) {
      if (own[t] != cur) {
        cur = own[t];
#pragma unroll
        for (int j = 0; j < R / 8; ++j) b[0][j] = load16(b_stack + ((long)cur * V + v) * R + j * 8);
      }
    }
    float acc = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r)
      acc = __builtin_fmaf(__bfloat162float(b[AHEAD ? t : 0][r / 8].data[r % 8]),
                           sums[t][p * R + r], acc);
    o[(long)t * out_w] = __float2bfloat16(__bfloat162float(was[t]) + acc * scale[t]);
  }
}

template <int R>
void launch_expand(__hip_bfloat16* out, const float* tmp, const __hip_bfloat16* b,
                   const int* slots, const float* scales, const LoraCols& cols, int T, int PR,
                   int V, int out_w, int cuts, hipStream_t stream) {
  auto go = [&](auto kernel, int tokens) {
    hipLaunchKernelGGL(kernel, dim3((V + 255) / 256, (T + tokens - 1) / tokens), dim3(256), 0,
                       stream, out, tmp, b, slots, scales, cols, T, PR, V, out_w, cuts);
  };
  // Tokens a workgroup: few keep the chip full, many share the sums' way through LDS and
  // the rows of B.  Rank 16, by 256-column tiles of all tokens (us at 2, 4, 8, 16 tokens):
  // 976 3.7 4.4 5.6 8.2, 6832 7.0 5.9 6.6 9.7, 14336 12.1 9.6 8.7 11.5, 67200 67 50 41 44,
  // 229376 157 123 106 102; ranks 8 and 64 cross at the same places.
  // The form for few tokens, us there | here at two tokens: rank 16, 8 cuts of K, 976 tiles 3.1 |
  // 3.7, 2560 3.7 | 4.0, 3840 4.5 | 4.7, 4800 5.3 | 5.0 (at four); 4 cuts, 1600 3.3 | 3.5, 2400 3.9 |
  // 3.7; rank 64, 8 cuts, 976 6.7 | 7.2, 1600 7.0 | 7.4, 2400 9.3 | 9.4; 4 cuts, 1200 7.0 | 6.8; rank
  // 8, 16384 tiles 9.9 | 6.4 (at eight).
  const long tiles = (V + 255L) / 256 * T;
  if (tiles <= (R <= 16 ? 2048 : 1024) * (cuts >= 8 ? 2 : 1)) go(lora_expand_few_kernel<R>, 2);
  else if (tiles <= 2560) go(lora_expand_tile_kernel<R, 2>, 2);
  else if (tiles <= 8192) go(lora_expand_tile_kernel<R, 4>, 4);
  else if (tiles <= 98304) go(lora_expand_tile_kernel<R, 8>, 8);
  else go(lora_expand_tile_kernel<R, 16>, 16);
}

// What becomes of a product together with its deltas, for all of its columns: the sum of its
// f32 parts (or the product itself, bf16) plus the deltas, and with GATE the first half's silu
// times the second.  One launch for what were two or three (a merge, expand, a gate), results
// rounded once.  grid (ceil(columns of out / 256), ceil(T / TOKENS)); bound as expand is.
// 61 tokens of 4 adapters of rank 16: merge and expand into 4096 columns 3.9 + 4.0 -> 5.0 us,
// expand into 28672 and the gate 8.5 -> 7.5.  With the gate two columns' rows of B are held, from
// rank 32 on at the cost of waves (136 to 256 registers): engine/lora.py says up to how many tokens
// it is the faster way.
template <int R, int TOKENS, bool GATE, bool FEW>
__global__ __launch_bounds__(256) void lora_finish_kernel(
    __hip_bfloat16* __restrict__ out,            // [T, GATE ? W / 2 : W]
    const __hip_bfloat16* __restrict__ base,     // [T, W] (parts == 0)
    const float* __restrict__ part,              // [parts, T, W]
    const float* __restrict__ tmp,               // [cuts, T, PR]
    const __hip_bfloat16* __restrict__ b_stack,  // [L, V, R]
    const int* __restrict__ slots, const float* __restrict__ scales, const LoraCols cols,
    const int T, const int PR, const int V, const int W, const int cuts, const int parts) {
  constexpr int H = GATE ? 2 : 1;
  constexpr bool AHEAD = FEW && TOKENS * R * H <= 64;
  __shared__ float sums[TOKENS][3 * R];
  const int OW = W / H, t0 = blockIdx.y * TOKENS, n = blockIdx.x * 256 + threadIdx.x;
  const int tokens = min(TOKENS, T - t0);
  int own[TOKENS];
#pragma unroll
  for (int t = 0; t < TOKENS; ++t)
    own[t] = __builtin_amdgcn_readfirstlane(t < tokens ? slots[t0 + t] : -1);
  // the projection and the row of B of this thread's columns, -1: none
  int proj[H], row[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const int c = n + h * OW;
    proj[h] = 0;
    row[h] = -1;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const int v = c - cols.shift[p];
      if (v >= (p > 0 ? cols.end[p - 1] : 0) && v < cols.end[p]) {
        proj[h] = p;
        row[h] = v;
      }
    }
    if (n >= OW) row[h] = -1;
  }
  float sum[TOKENS][H];
  Vec16<__hip_bfloat16> b[AHEAD ? TOKENS : 1][H][R / 8];
  float scale[TOKENS];
#pragma unroll
  for (int t = 0; t < TOKENS; ++t)
#pragma unroll
    for (int h = 0; h < H; ++h) {
      sum[t][h] = 0.f;
      if (n >= OW || t >= tokens) continue;
      const long at = (long)(t0 + t) * W + n + h * OW;
      if (parts == 0) {
        sum[t][h] = __bfloat162float(base[at]);
      } else {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = part[(long)min(i, parts - 1) * T * W + at];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i < parts) sum[t][h] += v[i];
      }
      if constexpr (AHEAD) {
        if (own[t] >= 0 && row[h] >= 0)
#pragma unroll
          for (int j = 0; j < R / 8; ++j)
            b[t][h][j] = load16(b_stack + ((long)own[t] * V + row[h]) * R + j * 8);
      }
    }
#pragma unroll
  for (int t = 0; t < TOKENS; ++t) scale[t] = own[t] >= 0 ? scales[own[t]] : 0.f;
  // (tokens without an adapter: whatever is there, which is not used)
  add_cuts<R, TOKENS, FEW>(sums, tmp, T, t0, tokens, PR, cuts);
  __syncthreads();
  if (n >= OW) return;
  int cur = -1;
#pragma unroll
  for (int t = 0; t < TOKENS; ++t) {
    if (t >= tokens) continue;
    if (own[t] >= 0) {
      if constexpr (!AHEAD) {
        if (own[t] != cur) {
          cur = own[t];
#pragma unroll
          for (int h = 0; h < H; ++h)
            if (row[h] >= 0)
#pragma unroll
              for (int j = 0; j < R / 8; ++j)
                b[0][h][j] = load16(b_stack + ((long)cur * V + row[h]) * R + j * 8);
        }
      }
#pragma unroll
      for (int h = 0; h < H; ++h) {
        if (row[h] < 0) continue;
        float acc = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r)
          acc = __builtin_fmaf(__bfloat162float(b[AHEAD ? t : 0][h][r / 8].data[r % 8]),
                               sums[t][proj[h] * R + r], acc);
        sum[t][h] += acc * scale[t];
      }
    }
    float y = sum[t][0];
    if constexpr (GATE) y = y / (1.f + __expf(-y)) * sum[t][H - 1];
    out[(long)(t0 + t) * OW + n] = __float2bfloat16(y);
  }
}

// The same by the matrix unit, 16 tokens of one adapter (or of none) at a time: products of B's
// rows, which are bf16, and the tokens' f32 sums of the shrink in three terms of eight bits, which
// are all 24 of them, with sums in f32.  Bound by the reads and writes of the product; a wave takes
// 32 columns at a time, its lanes eight neighbours of a token each.  us with the shrink, a column a
// thread | here: 948 x 28672 rank 64 in place 314 | 69, 868 x 28672 rank 32 119 | 50, 1582 x 28672 rank 8
// 107 | 63, 359 x 2048 rank 64 21.9 | 15.5, 107 x 4096 rank 64 15.8 | 13.6; with the gate 2048 x 28672 rank
// 8 151 | 104, 1000 x 28672 rank 16 106 | 61.
// grid (ceil(columns of out / (128 chunks)), windows x groups_of(kWindow, L + 1))
template <int R, bool GATE>
__global__ __launch_bounds__(256) void lora_finish_tile_kernel(
    __hip_bfloat16* out,                         // [T, GATE ? W / 2 : W]
    const __hip_bfloat16* base,                  // [T, W] (parts == 0); may be out
    const float* __restrict__ part,              // [parts, T, W]
    const float* __restrict__ tmp,               // [cuts, T, PR]
    const __hip_bfloat16* __restrict__ b_stack,  // [L, V, R]
    const int* __restrict__ slots, const float* __restrict__ scales, const LoraCols cols,
    const int T, const int L, const int PR, const int V, const int W, const int cuts,
    const int parts, const int chunks) {
  using lora::bf16x8_t;
  using lora::f32x4_t;
  constexpr int H = GATE ? 2 : 1, KS = (R + 31) / 32, PAD = 3 * R + 8, WINDOW = lora::kWindow;
  __shared__ __align__(16) unsigned short terms[3][16][PAD];   // of the tokens' sums
  __shared__ int groups[4][16];
  const int OW = W / H;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, quad = lane >> 4;
  const int per = lora::groups_of(WINDOW, L + 1), t0 = blockIdx.y / per * WINDOW;

  // the group: as in the shrink, but that -1 is an adapter too
  int first = blockIdx.y % per, slot, slot_of[WINDOW / 64];
#pragma unroll
  for (int i = 0; i < WINDOW / 64; ++i)
    slot_of[i] = t0 + i * 64 + lane < T ? max(slots[t0 + i * 64 + lane], -1) : -2;
  for (slot = -1; slot < L; ++slot) {
    int n = 15;
#pragma unroll
    for (int i = 0; i < WINDOW / 64; ++i) n += __popcll(__ballot(slot_of[i] == slot));
    if (first < n / 16) break;
    first -= n / 16;
  }
  if (slot == L) return;
  first *= 16;
  int* group = groups[wave];
  int found = 0;
#pragma unroll
  for (int i = 0; i < WINDOW / 64; ++i) {
    const unsigned long long has = __ballot(slot_of[i] == slot);
    const int at = found + __popcll(has & ((1ull << lane) - 1)) - first;
    if (slot_of[i] == slot && at >= 0 && at < 16) group[at] = t0 + i * 64 + lane;
    found += __popcll(has);
  }
  const int tokens = min(found - first, 16);
  // other lanes of this wave read it: LDS keeps a wave's order, the compiler has to
  asm volatile("" ::: "memory");
  const int own = group[min(col, tokens - 1)];

  // projections with columns among [c, c + n)
  auto meets = [&](int p, int c, int n) {
    const int v0 = p > 0 ? cols.end[p - 1] : 0;
    return v0 < cols.end[p] && c < cols.end[p] + cols.shift[p] && c + n > v0 + cols.shift[p];
  };
  const int c_wg = blockIdx.x * chunks * 128;
  int lo = 3, hi = -1;
  if (slot >= 0)
#pragma unroll
    for (int p = 0; p < 3; ++p)
      if (meets(p, c_wg, min(chunks * 128, OW - c_wg)) ||
          (GATE && meets(p, c_wg + OW, min(chunks * 128, OW - c_wg)))) {
        lo = min(lo, p);
        hi = max(hi, p);
      }
  if (base == out && hi < 0) return;

  float sum[H][8];
  auto load = [&](int c) {
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const long at = (long)own * W + c + h * OW + quad * 8;
      if (parts == 0) {
        const Vec16<__hip_bfloat16> v = load16(base + at);
#pragma unroll
        for (int i = 0; i < 8; ++i) sum[h][i] = __bfloat162float(v.data[i]);
        continue;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) sum[h][i] = 0.f;
      for (int p0 = 0; p0 < parts; p0 += 4) {
        f32x4_t v[4][2];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const f32x4_t* from = reinterpret_cast<const f32x4_t*>(
              part + (long)min(p0 + p, parts - 1) * T * W + at);
          v[p][0] = from[0];
          v[p][1] = from[1];
        }
#pragma unroll
        for (int p = 0; p < 4; ++p)
          if (p0 + p < parts)
#pragma unroll
            for (int i = 0; i < 8; ++i) sum[h][i] += v[p][i / 4][i % 4];
      }
    }
  };
  float scale = 0.f;
  if (hi >= 0) {
    scale = scales[slot];
    // the shrink's sums of the tokens: of the projections that are met
    const int width = (hi - lo + 1) * R;
    for (int i = threadIdx.x; i < 16 * width; i += 256) {
      const int m = i / width, r = lo * R + i % width;
      const float* from = tmp + (long)group[min(m, tokens - 1)] * PR + r;
      float s = 0.f;
      for (int q0 = 0; q0 < cuts; q0 += 4) {
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = from[(long)min(q0 + q, cuts - 1) * T * PR];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q0 + q < cuts) s += v[q];
      }
      // cut off, not rounded: infinity stays the first term, the others have its sign; none of a sum
      // that is not 0 is 0, which infinities in B would make NaN, but a least number
      const float sign = s, least = s == 0.f ? 0.f : FLT_MIN;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const unsigned bits = __float_as_uint(s);
        terms[k][m][r] =
            (k == 0 ? bits : __float_as_uint(copysignf(fmaxf(fabsf(s), least), sign))) >> 16;
        s = (bits & 0x7fffffff) == 0x7f800000 ? 0.f : s - __uint_as_float(bits & 0xffff0000);
      }
    }
    __syncthreads();
  }

  for (int u = 0; u < chunks; ++u) {
    const int c = c_wg + u * 128 + wave * 32;
    if (c >= OW) break;
    load(c);
    if (hi >= 0) {
      for (int p = lo; p <= hi; ++p) {
        const int v0 = p > 0 ? cols.end[p - 1] : 0;
        bf16x8_t x[KS][3];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int r = ks * 32 + quad * 8;
#pragma unroll
          for (int k = 0; k < 3; ++k)
            x[ks][k] = r < R ? *reinterpret_cast<const bf16x8_t*>(&terms[k][col][p * R + r])
                             : bf16x8_t{};
        }
#pragma unroll
        for (int h = 0; h < H; ++h) {
          if (!meets(p, c + h * OW, 32)) continue;
          f32x4_t acc[2] = {f32x4_t{}, f32x4_t{}};
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            // a lane's sums are of eight neighbouring columns
            const int v = c + h * OW + col / 4 * 8 + j * 4 + col % 4 - cols.shift[p];
            const bool in = v >= v0 && v < cols.end[p];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
              bf16x8_t w = bf16x8_t{};
              if (in && ks * 32 + quad * 8 < R)
                w = *reinterpret_cast<const bf16x8_t*>(b_stack + ((long)slot * V + v) * R +
                                                       ks * 32 + quad * 8);
#pragma unroll
              for (int k = 2; k >= 0; --k)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x[ks][k], acc[j], 0, 0, 0);
            }
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) {   // (an infinite sum is no zero beside the projection)
            const int v = c + h * OW + quad * 8 + i - cols.shift[p];
            if (v >= v0 && v < cols.end[p]) sum[h][i] += acc[i / 4][i % 4] * scale;
          }
        }
      }
    }
    if (col >= tokens) continue;
    union { __hip_bfloat16 h[8]; uint4 u; } o;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float y = sum[0][i];
      if constexpr (GATE) y = y / (1.f + __expf(-y)) * sum[H - 1][i];
      o.h[i] = __float2bfloat16(y);
    }
    *reinterpret_cast<uint4*>(out + (long)own * OW + c + quad * 8) = o.u;
  }
}

// Groups of 16 tokens that T tokens of L adapters, and some of none, leave at most
long finish_groups(int T, int L) {
  return T / lora::kWindow * (long)lora::groups_of(lora::kWindow, L + 1) +
         lora::groups_of(T % lora::kWindow, L + 1);
}

template <int R, bool GATE>
void launch_finish_tiles(__hip_bfloat16* out, const __hip_bfloat16* base, const float* part,
                         const float* tmp, const __hip_bfloat16* b, const int* slots,
                         const float* scales, const LoraCols& cols, int T, int L, int PR, int V,
                         int W, int cuts, int parts, hipStream_t stream) {
  const int OW = GATE ? W / 2 : W;
  const long groups = finish_groups(T, L), all = (OW + 127L) / 128 * groups;
  const int chunks = all > 8192 ? 4 : all > 4096 ? 2 : 1;   // of 128 columns, a workgroup
  hipLaunchKernelGGL((lora_finish_tile_kernel<R, GATE>),
                     dim3((OW + 128 * chunks - 1) / (128 * chunks), groups), dim3(256), 0, stream,
                     out, base, part, tmp, b, slots, scales, cols, T, L, PR, V, W, cuts, parts,
                     chunks);
}

template <int R, bool GATE>
void launch_finish(__hip_bfloat16* out, const __hip_bfloat16* base, const float* part,
                   const float* tmp, const __hip_bfloat16* b, const int* slots,
                   const float* scales, const LoraCols& cols, int T, int L, int PR, int V, int W,
                   int cuts, int parts, hipStream_t stream) {
  const int OW = GATE ? W / 2 : W;
  // (with the gate rank 64 is asked for where products are few: engine/lora.py, _GATE_TILES)
  if constexpr (!GATE || R < 64) {
    if (lora_tiles_win(T, L, R, W) && OW % 32 == 0) {
      launch_finish_tiles<R, GATE>(out, base, part, tmp, b, slots, scales, cols, T, L, PR, V, W,
                                   cuts, parts, stream);
      return;
    }
  }
  auto go = [&](auto kernel, int tokens) {
    hipLaunchKernelGGL(kernel, dim3((OW + 255) / 256, (T + tokens - 1) / tokens), dim3(256), 0,
                       stream, out, base, part, tmp, b, slots, scales, cols, T, PR, V, W, cuts,
                       parts);
  };
  // as in launch_expand, by what a thread has to do (many tokens: B is read where an adapter
  // begins, rank 8, 57344 tiles with the gate 39.7 -> 30.2 us)
  const long tiles = (W + 255L) / 256 * T;
  if (tiles <= 2560) go(lora_finish_kernel<R, 2, GATE, true>, 2);
  else if (tiles <= 8192) go(lora_finish_kernel<R, 4, GATE, true>, 4);
  else if (tiles <= 98304) go(lora_finish_kernel<R, 4, GATE, false>, 4);
  else go(lora_finish_kernel<R, 8, GATE, false>, 8);
}

// slot of every token: the place of its adapter's id among `ids`, or -1
struct LoraIds {
  int n, id[64];
};

__global__ __launch_bounds__(256) void lora_slots_kernel(int* __restrict__ slots,
                                                         const int* __restrict__ token_ids,
                                                         const LoraIds ids, const int T) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  const int id = token_ids[t];
  int s = -1;
  for (int i = 0; i < ids.n; ++i)
    if (ids.id[i] == id) s = i;
  slots[t] = s;
}

}  // namespace

void launch_lora_slots(int* slots, const int* token_ids, const int* ids, int n, int T,
                       hipStream_t stream) {
  LoraIds by_value{};
  by_value.n = n;
  for (int i = 0; i < n && i < 64; ++i) by_value.id[i] = ids[i];
  hipLaunchKernelGGL(lora_slots_kernel, dim3((T + 255) / 256), dim3(256), 0, stream, slots,
                     token_ids, by_value, T);
}

// Whether deltas of T tokens into W columns are added by the matrix unit: where the products are more
// than a launch's chain of loads, and than what every group that there may be, empty or not, takes for
// its columns, which grows with the adapters that it looks through.  us, a column a thread | matrix unit:
// 61 x 28672, 4 adapters of rank 16 13.0 | 13.2, 61 x 6144, 4 of 64 19.1 | 17.3, 436 x 2048, one of 32 8.5 |
// 9.0, 872 x 4096, 5 of 8 12.6 | 13.5; 1069 x 2048, 32 of 64 in four runs 38.6 | 41.3; 60 of 32, 200 x 6144
// 14.8 | 35.3, 599 x 2048 20.0 | 38.5; taken: 109 x 4096, 4 of 64 12.6 | 11.9, 458 x 28672, 60 of 64
// 243 | 126.  Of 1205 sizes of 1 to 60 adapters none is slower by more than 3 %, and of what all would
// gain 4 % is left.
bool lora_tiles_win(int T, int L, int R, int W) {
  return (long)T * W * R >= 28000000 + 7 * (L + 4) * finish_groups(T, L) * W;
}

// Workgroups K is cut over: enough for one a CU, four steps a wave at least (K 14336, rank
// 16, 61 tokens: 29.5 us uncut, 6.1 in 8, 4.2 in 16; K 4096: 12.5, 3.7, 3.1, and as much
// again in expand's sums; 2048 tokens: 23 us uncut and in 16).
int lora_shrink_cuts(int T, int K) {
  const int tiles = (T + 15) / 16;
  int cuts = (256 + tiles - 1) / tiles;
  if (cuts > 16) cuts = 16;
  const int most = K >= 1024 ? K / (32 * kShrinkWaves * 4) : 1;
  return cuts < most ? cuts : most;
}

// tmp [cuts, T, PR] = the tokens' rows of A x, in parts
void launch_lora_shrink_tiles(float* tmp, const __hip_bfloat16* x, const __hip_bfloat16* a,
                              const int* slots, int T, int L, int PR, int K, int cuts,
                              hipStream_t stream) {
  auto shrink = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(cuts, L, (T + 15) / 16), dim3(64 * kShrinkWaves), 0, stream,
                       tmp, x, a, slots, T, PR, K);
  };
  const int tiles = (PR + 15) / 16;
  if (tiles <= 1) shrink(lora_shrink_tile_kernel<1>);
  else if (tiles <= 2) shrink(lora_shrink_tile_kernel<2>);
  else if (tiles <= 3) shrink(lora_shrink_tile_kernel<3>);
  else if (tiles <= 4) shrink(lora_shrink_tile_kernel<4>);
  else if (tiles <= 6) shrink(lora_shrink_tile_kernel<6>);
  else if (tiles <= 8) shrink(lora_shrink_tile_kernel<8>);
  else shrink(lora_shrink_tile_kernel<12>);
}

// R in {8, 16, 32, 64}, PR = projections * R; tmp [cuts, T, PR]
void launch_lora_tiles(__hip_bfloat16* out, float* tmp, const __hip_bfloat16* x,
                       const __hip_bfloat16* a, const __hip_bfloat16* b, const int* slots,
                       const float* scales, const LoraCols& cols, int T, int L, int R, int PR,
                       int V, int K, int out_w, int cuts, hipStream_t stream) {
  launch_lora_shrink_tiles(tmp, x, a, slots, T, L, PR, K, cuts, stream);
  const bool tiles = lora_tiles_win(T, L, R, V) && out_w % 32 == 0 &&
                     reinterpret_cast<uintptr_t>(out) % 16 == 0;
#define EXPAND(RR)                                                                            \
  if (tiles)                                                                                  \
    launch_finish_tiles<RR, false>(out, out, nullptr, tmp, b, slots, scales, cols, T, L, PR,  \
                                   V, out_w, cuts, 0, stream);                                \
  else                                                                                        \
    launch_expand<RR>(out, tmp, b, slots, scales, cols, T, PR, V, out_w, cuts, stream)
  switch (R) {
    case 8: EXPAND(8); break;
    case 16: EXPAND(16); break;
    case 32: EXPAND(32); break;
    default: EXPAND(64);
  }
#undef EXPAND
}

// out = the product (bf16 base, or parts > 0 f32 parts [parts, T, W], at most 8) and its deltas,
// gated: silu of the first half of the columns times the second
void launch_lora_finish(__hip_bfloat16* out, const __hip_bfloat16* base, const float* part,
                        const float* tmp, const __hip_bfloat16* b, const int* slots,
                        const float* scales, const LoraCols& cols, int T, int L, int R, int PR,
                        int V, int W, int cuts, int parts, bool gated, hipStream_t stream) {
#define FINISH(RR)                                                                             \
  if (R == RR && gated)                                                                        \
    launch_finish<RR, true>(out, base, part, tmp, b, slots, scales, cols, T, L, PR, V, W,      \
                            cuts, parts, stream);                                                    \
  else if (R == RR)                                                                            \
    launch_finish<RR, false>(out, base, part, tmp, b, slots, scales, cols, T, L, PR, V, W,     \
                             cuts, parts, stream)
  FINISH(8);
  FINISH(16);
  FINISH(32);
  FINISH(64);
#undef FINISH
}

#define INSTANTIATE_LORA(T)                                                  \
  template void launch_lora_shrink<T>(float*, const T*, const T*,            \
                                      const int*, int, int, int,             \
                                      hipStream_t);                          \
  template void launch_lora_expand<T>(T*, const float*, const T*,            \
                                      const int*, const float*, int, int,    \
                                      int, int, int, hipStream_t);

INSTANTIATE_LORA(float)
INSTANTIATE_LORA(__hip_bfloat16)
INSTANTIATE_LORA(__half)
