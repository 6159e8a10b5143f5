// Products of more than 64 rows in bf16, y[m, n] = sum_k x[m, k] W[n, k], with long K:
// block_gemm.h's tiles of 128 x 128, K cut over workgroups until there are two a CU, the
// parts' f32 sums added by a second launch.
//
// Bound, up to some 200 rows, by the bytes of W; the library's product of these shapes cuts
// K less and leaves most of the chip idle.  us in a captured graph over weights that are
// not in the caches (library -> here), N x K:
//   4096 x 14336: 65 rows 48.6 -> 40.8, 128 75 -> 40, 256 63 -> 53, 512 89 -> 85
//   8192 x 28672: 65 rows 193 -> 103, 128 203 -> 123, 256 317 -> 171
//   10240 x 8192: 128 rows 59 -> 50, 256 89 -> 67;  8192 x 8192: 48 -> 41, 76 -> 55

#include "block_gemm.h"

namespace {

using block_gemm::Block;
using block_gemm::f32x4_t;

constexpr int BM = 128, BN = 128, WM = 2, WN = 2;

// grid (tiles of y, parts of K); part [parts, M, N] (gridDim.y > 1); depth: K of a part
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_block_kernel(
    __hip_bfloat16* __restrict__ y, float* __restrict__ part,
    const __hip_bfloat16* __restrict__ x, const __hip_bfloat16* __restrict__ w, const int M,
    const int N, const int K, const int depth) {
  using B = Block<BM, BN, WM, WN, 2>;
  __shared__ __align__(16) char lds[B::kLds];
  // neighbours in a run of blocks that one XCD gets share their columns of W
  const int m_tiles = (M + BM - 1) / BM, blocks = m_tiles * (N / BN);
  const int per_xcd = (blocks + 7) / 8, slot = blockIdx.x / 8;
  const int id = (blockIdx.x % 8) * per_xcd + slot;
  if (slot >= per_xcd || id >= blocks) return;
  const int m0 = id % m_tiles * BM, n0 = id / m_tiles * BN, k0 = blockIdx.y * depth;

  f32x4_t acc[B::kTM][B::kTN];
#pragma unroll
  for (int i = 0; i < B::kTM; ++i)
#pragma unroll
    for (int j = 0; j < B::kTN; ++j) acc[i][j] = f32x4_t{};
  const unsigned row_bytes = K * 2;
  // rows past M: the last one, whose results are not written
  B::run(acc, lds, reinterpret_cast<const char*>(x + (long)m0 * K + k0),
         reinterpret_cast<const char*>(w + (long)n0 * K + k0), min(depth, K - k0),
         [&](int r) { return min(r, M - 1 - m0) * row_bytes; },
         [&](int r) { return r * row_bytes; });

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, quad = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
#pragma unroll
  for (int i = 0; i < B::kTM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + (wm * B::kTM + i) * 16 + quad * 4 + r;
      if (m >= M) continue;
      const long at = (long)m * N + n0 + wn * B::kTN * 16 + col;
#pragma unroll
      for (int j = 0; j < B::kTN; ++j) {
        if (gridDim.y > 1)
          part[blockIdx.y * ((long)M * N) + at + j * 16] = acc[i][j][r];
        else
          y[at + j * 16] = __float2bfloat16(acc[i][j][r]);
      }
    }
}

}  // namespace

void launch_gemm_merge(__hip_bfloat16* y, const float* part, long plane, int parts, bool gated,
                       hipStream_t stream);

// Workgroups that K is cut over (each leaves a part of the result in f32): as many as make
// two a CU, of eight tiles of 64 inputs at least.
int gemm_block_parts(int M, int N, int K) {
  const int blocks = (M + BM - 1) / BM * (N / BN);
  int parts = 512 / (blocks > 0 ? blocks : 1);
  if (parts > 8) parts = 8;
  if (parts > K / 512) parts = K / 512;
  if (parts <= 1) return 1;
  const int depth = (K / 64 + parts - 1) / parts;   // no part is empty
  return (K / 64 + depth - 1) / depth;
}

// N % 128 == 0, K % 64 == 0, 128 rows of x and of W inside 4 GB
void launch_gemm_block(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                       const __hip_bfloat16* w, int M, int N, int K, int parts,
                       hipStream_t stream) {
  const int blocks = (M + BM - 1) / BM * (N / BN);
  const int depth = (K / 64 + parts - 1) / parts * 64;
  hipLaunchKernelGGL(gemm_block_kernel, dim3((blocks + 7) / 8 * 8, parts), dim3(64 * WM * WN), 0,
                     stream, y, part, x, w, M, N, K, depth);
  if (parts > 1) launch_gemm_merge(y, part, (long)M * N, parts, false, stream);
}
