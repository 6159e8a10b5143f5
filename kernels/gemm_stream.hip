// Products of few rows with a whole weight matrix (decode, M <= 64; a single row with bf16
// or 4-bit weights: gemm_row.hip):
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
// and the scale is doubled.
//
// Measured against the kernels before (barriers around 64-input chunks, weights rounded
// to bf16 with their scale, a merge launch for every matrix), us a product with the
// merge where there is one:
//   23 rows, 14336 x 4096 gated 55.2 -> 43.4; the mean of 6144 x 4096, 4096 x 4096 and
//     4096 x 14336 23.9 -> 17.5 (a llama-3-8b layer reads W at 4.5 TB/s);
//   61 rows, the mean of these three and 28672 x 4096: 38.1 -> 30;

#include "gemm_stream.h"

using namespace gemm_stream;

namespace {

// y = the sum of the workgroups' parts, four neighbours a thread (M * N % 4 == 0)
template <bool GATED>
__global__ __launch_bounds__(256) void gemm_stream_merge_kernel(
    __hip_bfloat16* __restrict__ y, const float* __restrict__ part, const long plane,
    const int parts) {
  const long at = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (at >= plane) return;
  f32x4_t a{}, b{};
  for (int p = 0; p < parts; ++p) {
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
  if (gated)
    hipLaunchKernelGGL(gemm_stream_merge_kernel<true>, grid, dim3(256), 0, stream, y, part, plane,
                       parts);
  else
    hipLaunchKernelGGL(gemm_stream_merge_kernel<false>, grid, dim3(256), 0, stream, y, part,
                       plane, parts);
}

namespace {

// How a product is cut (waves along N x waves along K, workgroups along K).  The lines
// are where they measured fastest (us; bf16 unless said; N x K):
//   up to 16 rows of x, x is a small part of what is read and waves work alone:
//     4096 x 4096: 1x8 8.1, 1x4 9.5; 14336 x 4096 gated: 1x4 39.8, 1x8 42.0.
//   17..32, plain: 4096 x 4096: 1x8 11.2, 4x2 over 4 12.1; 4096 x 14336: 27.4, 25.4;
//     8192 x 8192: 4x2 over 2 30.4, 2x4 31.4; 28672 x 4096 int8: 4x2 27.3, 4x1 30.9.
//     gated: 14336 x 4096: 2x2 43.4, 1x4 45.5, 4x1 47.5; 28672 x 8192: 4x1 158, 2x2 171.
//   33..64, every wave's own copy of x would cost more than W: 4096 x 14336: 4x2 over 4
//     34.9, 1x8 43.5; 2048 x 2048: 1x8 9.4, 4x2 10.3; 28672 x 4096: int8 4x2 42, 8x1 over
//     2 45, 4 bits 8x1 over 2 41, 4x2 47 (more of x is turned per weight);
//     8192 x 28672: 4x2 over 4 93, over 2 109.  gated: 14336 x 4096: 2x2 48.4, 4x2 49.7;
//     28672 x 8192: 4x1 158, 2x2 189; 8192 x 2048: 2x4 18.0, 2x2 21.5.
enum class Cut { kWave8, kWave4, kShare22, kShare24, kShare41, kShare42, kShare81 };

Cut cut_of(int qbits, int M, int N, int K, bool gated) {
  if (M <= 16) return N / 16 < 512 ? Cut::kWave8 : Cut::kWave4;
  if (gated) {
    if (K >= 8192) return Cut::kShare41;
    return K < 4096 && M > 32 ? Cut::kShare24 : Cut::kShare22;
  }
  if ((long)N * K <= 1L << (M <= 32 ? 24 : 23)) return Cut::kWave8;
  if (qbits == 4 && M > 32 && N >= 16384 && K >= 4096) return Cut::kShare81;
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

// Workgroups that K is cut over besides the waves (each leaves a part of the result):
// as many as make one a CU, two where K is long and the columns are many.  A function of
// shapes.
int gemm_stream_parts(int qbits, int M, int N, int K, bool gated) {
  const Cut cut = cut_of(qbits, M, N, K, gated);
  if (gated || (cut != Cut::kShare42 && cut != Cut::kShare81)) return 1;
  const int wgs = N / (cut == Cut::kShare81 ? 128 : 64);
  const int want = M > 32 && N >= 8192 && K >= 8192 ? 512 : 256;
  int parts = (want + wgs - 1) / wgs;
  if (parts > 8) parts = 8;
  const int most = K / 1024 > 0 ? K / 1024 : 1;   // four tiles of 128 a wave at least
  return parts < most ? parts : most;
}

bool gemm_row_fits(int qbits, int K);
void launch_gemm_row(__hip_bfloat16* y, const __hip_bfloat16* x, const void* w,
                     const float* scale, int qbits, int N, int K, bool gated,
                     hipStream_t stream);

// M <= 64, N % 128 == 0, K % 64 == 0 (rounded weights: K % 128 == 0)
void launch_gemm_stream(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                        const __hip_bfloat16* w, int M, int N, int K, int parts,
                        hipStream_t stream) {
  if (M == 1 && gemm_row_fits(16, K))
    launch_gemm_row(y, x, w, nullptr, 16, N, K, false, stream);
  else
    launch_q<16, false>(y, part, x, w, nullptr, M, N, K, parts, stream);
}

void launch_gemm_stream_gated(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                              const __hip_bfloat16* w13, int M, int I, int K, int parts,
                              hipStream_t stream) {
  if (M == 1 && gemm_row_fits(16, K))
    launch_gemm_row(y, x, w13, nullptr, 16, I, K, true, stream);
  else
    launch_q<16, true>(y, part, x, w13, nullptr, M, I, K, parts, stream);
}

void launch_gemm_stream_q(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                          const unsigned char* wq, const float* scale, int qbits, int M, int N,
                          int K, int parts, hipStream_t stream) {
  if (M == 1 && gemm_row_fits(qbits, K))
    launch_gemm_row(y, x, wq, scale, qbits, N, K, false, stream);
  else if (qbits == 8)
    launch_q<8, false>(y, part, x, wq, scale, M, N, K, parts, stream);
  else
    launch_q<4, false>(y, part, x, wq, scale, M, N, K, parts, stream);
}
