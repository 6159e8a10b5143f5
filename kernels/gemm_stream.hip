// Products of few rows with a whole weight matrix (decode, M <= 64; a single row:
// gemm_row.hip; aligned bf16 of more than 8 rows, where they are faster: the tiles of
// gemm_ring.hip):
//   y[m, n] = sum_k x[m, k] W[n, k],  or  silu(x Wg^T) * (x Wu^T) for W = [Wg; Wu],
// with W in bf16, in int8 (a scale per row) or in 4 bits (offset 8, a scale per row
// and 128 inputs).
//
// Bound by the bytes of W.  A workgroup owns 16 to 64 rows of W (of both halves in
// the gated form) and cuts K over its waves in turns.  A wave takes a tile of its rows
// (whole 64 to 256 byte runs, read once: nontemporal) and of x through registers into
// LDS, two tiles ahead of the one it works on, and gets them back in the layout of
// v_mfma_f32_16x16x32_bf16's operands; 16-byte chunks are swizzled by row against bank
// conflicts.  Up to 16 rows of x waves work alone, without a barrier, and add up inside
// the workgroup: no second launch, and 4096 rows of W still fill the chip.  With more
// rows of x the waves along N share its tile (see cut_of).  A result has a W row per
// lane and four x rows in its registers, so that a row's scale is one multiplication.
//
// Rounded weights enter the product as whole numbers (exact in bf16) and the scales are
// applied to 32-bit sums, per group of 128 inputs or once at the end.  A 4-bit weight
// becomes 8 + n/2 by two logical operations a pair (n in the upper bits of a bf16
// mantissa); x is put in the order that this leaves the weights in, -12 times the sum
// of x, which the matrix unit adds by a constant operand, takes the offset out again
// and the scale is doubled.  (An infinite x, or one above 2^123, makes its row NaN there.)
//
// Measured against the kernels before (barriers around 64-input chunks, weights rounded
// to bf16 with their scale, a merge launch for every matrix), us a product with the
// merge where there is one:
//   23 rows, 14336 x 4096 gated 55.2 -> 43.4; the mean of 6144 x 4096, 4096 x 4096 and
//     4096 x 14336 23.9 -> 17.5 (a llama-3-8b layer reads W at 4.5 TB/s);
//   61 rows, the mean of these three and 28672 x 4096: 38.1 -> 30.
// (In bf16 the tiles have taken over from there at 23 and 61 rows, in rounded weights past 32 rows, and
// fewer where the matrix is large, the panels of gemm_block_q.hip; up to 16 rows, at short K, for
// small matrices and for rounded weights' operands off a 16-byte boundary these kernels are what runs.)

#include "gemm_stream.h"

using namespace gemm_stream;

namespace {

// y = the sum of the workgroups' parts, four neighbours a thread (M * N % 4 == 0)
// KNOWN: parts, all of them asked for at once; 0: any
template <bool GATED, int KNOWN>
__global__ __launch_bounds__(256) void gemm_stream_merge_kernel(
    __hip_bfloat16* __restrict__ y, const float* __restrict__ part, const long plane,
    const int parts) {
  const long at = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (at >= plane) return;
  f32x4_t a{}, b{};
  if constexpr (!GATED && KNOWN > 0) {
    f32x4_t v[KNOWN];
#pragma unroll
    for (int p = 0; p < KNOWN; ++p)
      v[p] = *reinterpret_cast<const f32x4_t*>(part + p * plane + at);
#pragma unroll
    for (int p = 0; p < KNOWN; ++p) a += v[p];
  } else for (int p = 0; p < parts; ++p) {
    a += *reinterpret_cast<const f32x4_t*>(part + p * (GATED ? 2 : 1) * plane + at);
    if (GATED) b += *reinterpret_cast<const f32x4_t*>(part + (p * 2 + 1) * plane + at);
  }
  union { __hip_bfloat16 h[4]; uint2 u; } o;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    o.h[r] = __float2bfloat16(GATED ? a[r] / (1.f + __expf(-a[r])) * b[r] : a[r]);
  *reinterpret_cast<uint2*>(y + at) = o.u;
}

}  // namespace

// y = the sum of parts of a product (of silu of the first half times the second)
void launch_gemm_merge(__hip_bfloat16* y, const float* part, long plane, int parts, bool gated,
                       hipStream_t stream) {
  const dim3 grid((plane / 4 + 255) / 256);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, y, part, plane, parts);
  };
  if (gated) return go(gemm_stream_merge_kernel<true, 0>);
  // Few rows are a chain of loads, which is one long if all parts are asked for at once; many are
  // bytes.  With their product, one part after the other | at once, us: 17 x 4096 (4096) 11.5 | 10.7, 23 x
  // 4096 (14336) 24.6 | 23.9, 61 x 4096 (4096) 13.1 | 12.6; 512 x 4096 (14336) 78.5 | 79.8.
  if (plane <= 1 << 20) switch (parts) {
    case 2: return go(gemm_stream_merge_kernel<false, 2>);
    case 3: return go(gemm_stream_merge_kernel<false, 3>);
    case 4: return go(gemm_stream_merge_kernel<false, 4>);
    case 5: return go(gemm_stream_merge_kernel<false, 5>);
    case 6: return go(gemm_stream_merge_kernel<false, 6>);
    case 7: return go(gemm_stream_merge_kernel<false, 7>);
    case 8: return go(gemm_stream_merge_kernel<false, 8>);
  }
  go(gemm_stream_merge_kernel<false, 0>);
}

namespace {

// How a product is cut (waves along N x waves along K, workgroups along K).  The lines
// are where they measured fastest (us from cold weights; bf16 unless said; N x K):
//   up to 16 rows of x, x is a small part of what is read and waves work alone:
//     4096 x 4096: 1x8 8.1, 1x4 9.5; 6144 x 4096: 1x4 13.2, 1x8 13.9; 5120 x 8192: 22.0,
//     25.0; 14336 x 4096 gated: 39.8, 42.0.
//   25 rows, plain: 4096 x 4096: 1x8 11.8, 4x2 over 4 12.4; 4096 x 14336: 28.6, 25.8;
//     8192 x 8192: 4x2 over 2 29.7, 1x8 34.6; 28672 x 4096 int8: 4x2 27.4, 4x1 31.0.
//   49 rows, every wave's own copy of x would cost more than W: 4096 x 14336: 4x2 over 8
//     32.6, 1x8 39.8; 2048 x 2048: 1x8 8.8, 4x2 over 4 9.9; 4 bits, where more of x is
//     turned per weight: 28672 x 4096: 8x1 over 2 44.3, 4x2 60; 8192 x 8192: 8x1 over 8
//     30.1, 4x2 over 2 35.9.
//   gated, 25 | 49 rows, by how many columns there are to share out (a whole layer's to an
//   eighth of one's):
//     28672 x 8192: 4x1 156 | 157, 2x2 173 | 191; 14336 x 8192: 2x2 79 | 91, 4x1 89 | 119;
//     14336 x 4096: 2x2 42.6 | 47.8, 4x1 47.7 | 62;
//     7168 x 4096: 1x4 26.0 | 30.8, 2x4 27.1 | 28.6, 2x2 28.5 | 35.0; 8064 x 8192: 1x4 47.9
//     | 57.6, 2x4 54.9 | 57.7, 2x2 54 | 68; 5120 x 4096: 2x4 22.8 | 25.9, 1x4 24.2 | 28.9;
//     3584 x 8192: 1x8 27.2 | 31.2, 2x4 37 | 45, 4x1 68 | 104; 2048 x 2048: 9.4 | 12.1,
//     2x4 12.3 | 14.5;
//     1280 x 8192: 2x4 over 6 16.7 | 18.4, 1x8 21.2 | 27.2; 1792 x 4096: over 4 13.5 | 15.1,
//     14.1 | 17.3; 64 rows, 2560 x 8192: over 3 26.8, 1x8 32.1; 4096 x 14336: over 2 53, 62.
enum class Cut { kWave8, kWave4, kShare22, kShare24, kShare41, kShare42, kShare81 };

Cut cut_of(int qbits, int M, int N, int K, bool gated) {
  if (M <= 16) return N / 16 <= 256 ? Cut::kWave8 : Cut::kWave4;
  if (gated) {
    if (N >= 20480 && K >= 8192) return Cut::kShare41;
    if (N >= 12288) return Cut::kShare22;
    if (N > 4096) return M <= 32 && N >= 6144 ? Cut::kWave4 : Cut::kShare24;
    return (N <= 2048 ? K >= 4096 : M > 32 && K >= 3 * N) ? Cut::kShare24 : Cut::kWave8;
  }
  if ((long)N * K <= 1L << (M <= 32 ? 24 : 23)) return Cut::kWave8;
  if (qbits == 4 && M > 32 && (N >= 16384 ? K >= 4096 : N >= 8192 && K >= 8192))
    return Cut::kShare81;
  return Cut::kShare42;
}

template <int QB, int MT, bool GATED, int WN, int WK>
void launch_cut(__hip_bfloat16* y, float* part, const __hip_bfloat16* x, const void* w,
                const float* s, int M, int N, int K, int parts, hipStream_t stream) {
  constexpr int kCols = 16 * WN;   // of a workgroup; N is a multiple of 128
  static_assert(128 % kCols == 0, "whole workgroups");
  hipLaunchKernelGGL(
      (gemm_stream_kernel<QB, MT, 1, WN, WK, GATED ? moe::kSilu : moe::kPlain>),
      dim3(N / kCols, parts), dim3(64 * WN * WK), 0, stream, y, part, x, w, s, M, N, K);
}

template <int QB, int MT, bool GATED>
void launch_mt(__hip_bfloat16* y, float* part, const __hip_bfloat16* x, const void* w,
               const float* s, int M, int N, int K, int parts, hipStream_t stream) {
  const Cut cut = cut_of(QB, M, N, K, GATED);
  auto run = [&](auto launch) { launch(y, part, x, w, s, M, N, K, parts, stream); };
  if constexpr (MT == 1) {
    if (cut == Cut::kWave8) run(launch_cut<QB, MT, GATED, 1, 8>);
    else run(launch_cut<QB, MT, GATED, 1, 4>);
  } else if constexpr (GATED) {
    if (cut == Cut::kShare41) run(launch_cut<QB, MT, GATED, 4, 1>);
    else if (cut == Cut::kShare24) run(launch_cut<QB, MT, GATED, 2, 4>);
    else if (cut == Cut::kWave8) run(launch_cut<QB, MT, GATED, 1, 8>);
    else if (cut == Cut::kWave4) run(launch_cut<QB, MT, GATED, 1, 4>);
    else run(launch_cut<QB, MT, GATED, 2, 2>);
  } else if (cut == Cut::kWave8) {
    run(launch_cut<QB, MT, GATED, 1, 8>);
  } else {
    if constexpr (QB == 4) {
      if (cut == Cut::kShare81) run(launch_cut<QB, MT, GATED, 8, 1>);
      else run(launch_cut<QB, MT, GATED, 4, 2>);
    } else {
      run(launch_cut<QB, MT, GATED, 4, 2>);
    }
  }
  if (parts > 1) launch_gemm_merge(y, part, (long)M * N, parts, GATED, stream);
}

template <int QB, bool GATED>
void launch_q(__hip_bfloat16* y, float* part, const __hip_bfloat16* x, const void* w,
              const float* s, int M, int N, int K, int parts, hipStream_t stream) {
  if (M <= 16) launch_mt<QB, 1, GATED>(y, part, x, w, s, M, N, K, parts, stream);
  else if (M <= 32) launch_mt<QB, 2, GATED>(y, part, x, w, s, M, N, K, parts, stream);
  else launch_mt<QB, 4, GATED>(y, part, x, w, s, M, N, K, parts, stream);
}

}  // namespace

// Workgroups that K is cut over besides the waves (each leaves a part of the result), of four
// tiles of 128 a wave at least: what fills whole rounds of one workgroup a CU best, up to two
// rounds.  us, 25 | 49 rows, waves 4x2 over 2, 3, 4 workgroups: 6144 x 4096 (96 columns of
// workgroups) 15.4 18.7 17.1 | 20.3 20.4 19.3; 7168 x 8192 (112) 26.7 30.4 27.7 | 34.6 34.0
// 30.5; 10240 x 4096 (160) 24.3 21.3 22.5 | 27.2 23.3 29.1; 16384 x 2048 (256), over 1 and 2,
// 15.7 18.7 | 18.9 22.0.  Two rounds rather than one as full go with more rows of x, in 4 bits
// with fewer (8192 x 8192 over 2, 4: 28.5 22.7 | 35.9 37.7).  A function of shapes.
int gemm_stream_parts(int qbits, int M, int N, int K, bool gated) {
  const Cut cut = cut_of(qbits, M, N, K, gated);
  if (gated) {   // columns that are few are cut over as many workgroups as there are CUs
    const int fill = cut == Cut::kShare24 && N <= 4096 ? 256 / (N / 32) : 1;
    const int most = K / 1024 < 8 ? K / 1024 : 8;
    return fill < most ? fill : most > 0 ? most : 1;
  }
  if (cut != Cut::kShare42 && cut != Cut::kShare81) return 1;
  const int wgs = N / (cut == Cut::kShare81 ? 128 : 64);
  const bool two = wgs < 256 && (cut == Cut::kShare81 || (qbits == 4) == (M <= 32));
  int parts = 1, best = 0;
  for (int p = 1; p <= 8 && (p == 1 || (p <= K / 1024 && wgs * p <= 512)); ++p) {
    const int rounds = (wgs * p + 255) / 256, full = wgs * p / rounds;
    if (full > best || (full == best && two)) {
      parts = p;
      best = full;
    }
  }
  return parts;
}

bool gemm_row_fits(int K);
void launch_gemm_row(__hip_bfloat16* y, const __hip_bfloat16* x, const void* w,
                     const float* scale, int qbits, int N, int K, bool gated,
                     hipStream_t stream);

// M <= 64, N % 128 == 0, K % 64 == 0 (rounded weights: K % 128 == 0)
void launch_gemm_stream(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                        const __hip_bfloat16* w, int M, int N, int K, int parts,
                        hipStream_t stream) {
  if (M == 1 && gemm_row_fits(K))
    launch_gemm_row(y, x, w, nullptr, 16, N, K, false, stream);
  else
    launch_q<16, false>(y, part, x, w, nullptr, M, N, K, parts, stream);
}

void launch_gemm_stream_gated(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                              const __hip_bfloat16* w13, int M, int I, int K, int parts,
                              hipStream_t stream) {
  if (M == 1 && gemm_row_fits(K))
    launch_gemm_row(y, x, w13, nullptr, 16, I, K, true, stream);
  else
    launch_q<16, true>(y, part, x, w13, nullptr, M, I, K, parts, stream);
}

void launch_gemm_stream_q(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                          const unsigned char* wq, const float* scale, int qbits, int M, int N,
                          int K, int parts, hipStream_t stream) {
  // int8 of short K: a workgroup of gemm_row.hip has one segment of a row or less (us, here |
  // there: 768 x 768 2.7 | 3.0, 4096 x 1024 3.2 | 3.5, 2048 x 1024 3.0 | 3.2; 1024 x 2048
  // 3.7 | 3.2, 2048 x 2048 3.8 | 3.5)
  if (M == 1 && gemm_row_fits(K) && !(qbits == 8 && K <= 1024))
    launch_gemm_row(y, x, wq, scale, qbits, N, K, false, stream);
  else if (qbits == 8)
    launch_q<8, false>(y, part, x, wq, scale, M, N, K, parts, stream);
  else
    launch_q<4, false>(y, part, x, wq, scale, M, N, K, parts, stream);
}
