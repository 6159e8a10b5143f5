// Products of many rows, y[m, n] = sum_k x[m, k] W[n, k] or silu(x Wg^T) * (x Wu^T) for
// W = [Wg; Wu], in bf16: ring_gemm.h's loop over tiles of 64 to 256 rows of x, K cut over
// workgroups where the tiles are too few for the chip (the parts' f32 sums are added by a
// second launch).
//
// Up to some 250 rows these are bound by the bytes of W, above by the matrix unit; between,
// by how well tiles fill whole rounds of 256 CUs, so that the tile and the cut are chosen by
// a cost model (plan_of below).  us, the library (with its gate in a launch of its own; 4096 x
// 14336: our 128 x 128 tiles before) -> here, cold weights, rows x N x K:
//   gated 8192 x 14336 x 4096 1426 -> 1316; 2049 x 14336 x 4096 413 -> 382; 512 x 14336 x 4096
//     108 -> 96; 512 x 8192 x 2048 43 -> 35; 192 x 2048 x 2048 16 -> 10
//   plain 512 x 4096 x 14336 85 -> 70; 65 x 4096 x 14336 38 -> 29; 192 x 4096 x 4096 33 -> 20;
//     128 x 6144 x 4096 27 -> 20
// What did not pay: tiles of 256 x 128 beside 128 x 256 (within 1 %), five slots of 128 x 128
// (2 % here and there), 64 x 256.

#include "ring_gemm.h"
#include "moe_tiles.h"

namespace {

using ring_gemm::f32x4_t;

// grid (tiles of y, parts of K); part [parts, M, N] (gridDim.y > 1); depth: K of a part
template <int BM, int BN, int SLOTS, int OCC, bool GATED, int HINT = 0>
__global__ __launch_bounds__(256, OCC) void gemm_ring_kernel(
    __hip_bfloat16* __restrict__ y, float* __restrict__ part,
    const __hip_bfloat16* __restrict__ x, const __hip_bfloat16* __restrict__ w, const int M,
    const int N, const int K, const int depth) {
  using R = ring_gemm::Ring<BM, BN, 2, 2, SLOTS, HINT>;
  constexpr int COLS = GATED ? BN / 2 : BN;              // outputs of a block
  constexpr int OUT = GATED ? R::kTN / 2 : R::kTN;       // output tiles of a wave
  __shared__ __align__(16) char lds[R::kLds];
  // Each XCD has a run of neighbours: bands of up to eight tiles of rows, column by column,
  // so that the tiles that run at a time share rows of x and of W in its L2
  const int m_tiles = (M + BM - 1) / BM, n_tiles = N / COLS, blocks = m_tiles * n_tiles;
  const int per_xcd = (blocks + 7) / 8, slot = blockIdx.x / 8;
  const int id = (blockIdx.x % 8) * per_xcd + slot;
  if (slot >= per_xcd || id >= blocks) return;
  const int band = id / (8 * n_tiles), in = id % (8 * n_tiles), high = min(8, m_tiles - band * 8);
  const int m0 = (band * 8 + in % high) * BM, n0 = in / high * COLS, k0 = blockIdx.y * depth;

  f32x4_t acc[R::kTM][R::kTN];
  R::clear(acc);
  const unsigned row_bytes = K * 2;
  // rows past M: the last one, whose results are not written
  R::run(acc, lds, reinterpret_cast<const char*>(x + (long)m0 * K + k0),
         reinterpret_cast<const char*>(w + (long)n0 * K + k0), min(depth, K - k0),
         [&](int r) { return min(r, M - 1 - m0) * row_bytes; },
         [&](int r) {
           const int wave = r / (R::kTN * 16), at = r % (R::kTN * 16), half = at / (OUT * 16);
           const int col = at % (OUT * 16);
           return (half * N + wave * (OUT * 16) + (OUT > 1 ? R::out_col(col) : col)) * row_bytes;
         });

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, quad = lane >> 4, wm = wave / 2, wn = wave % 2;
#pragma unroll
  for (int i = 0; i < R::kTM; ++i) {
    const int m = m0 + (wm * R::kTM + i) * 16 + col;
    if (m >= M) continue;
    const long at = (long)m * N + n0 + wn * OUT * 16 + quad * (OUT > 1 ? 8 : 4);
    if constexpr (OUT == 1) {
      union { __hip_bfloat16 h[4]; uint2 u; } o;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o.h[r] = __float2bfloat16(moe::finish<moe::kSilu>(acc[i][0][r], acc[i][1][r], 0.f));
      *reinterpret_cast<uint2*>(y + at) = o.u;
    }
#pragma unroll
    for (int j = 0; j + 1 < OUT; j += 2) {
      if (!GATED && gridDim.y > 1) {
        float* to = part + blockIdx.y * ((long)M * N) + at + j * 16;
        *reinterpret_cast<f32x4_t*>(to) = acc[i][j];
        *reinterpret_cast<f32x4_t*>(to + 4) = acc[i][j + 1];
        continue;
      }
      union { __hip_bfloat16 h[8]; uint4 u; } o;
#pragma unroll
      for (int r = 0; r < 8; ++r)
        o.h[r] = __float2bfloat16(moe::finish<GATED ? moe::kSilu : moe::kPlain>(
            acc[i][j + r / 4][r % 4], acc[i][(GATED ? OUT : 0) + j + r / 4][r % 4], 0.f));
      *reinterpret_cast<uint4*>(y + at + j * 16) = o.u;
    }
  }
}

// A tile's form and what its time is made of, in us, fitted to some 2000 measured products
// (24 shapes of W of the presets and their shards, 17 to 8192 rows; standard deviation 8 to
// 12 %): the start, a workgroup's start and end and its tiles of 64 inputs, alone on its CU and
// in pairs, and a second launch for parts of K.
struct Form {
  int bm, bn, pairs;
  double start, own, one, two, merge, merge_mb, w_mb;
};
constexpr Form kForms[] = {
    {256, 256, 1, 0.0, 8.3, 1.13, 1.13, 4.1, 0.16, 0.24},
    {128, 256, 1, 0.0, 2.4, 0.76, 0.76, 4.4, 0.21, 0.21},
    {128, 128, 2, 1.5, 0.3, 0.48, 1.00, 3.9, 0.20, 0.21},
    {64, 128, 2, 2.3, 0.0, 0.34, 0.77, 3.2, 0.21, 0.20},
};
// The fifth form, 64 x 64 for up to 64 rows, is not fitted: few_rows below (gated: not cut).
constexpr int kFew = 4, kForm4Cols = 64;

struct Plan {
  int form, parts;
  double us;
};

// Up to 64 rows x is one tile and W comes by once: workgroups of 64 rows of W, as many as there
// are CUs (K cut), or two a CU where that leaves a quarter of them idle or K stays long, and W
// past the caches.  us, the streaming kernel | 64 x 128 by the model below | here, N x K, 24 |
// 64 rows: 28672 x 4096 44.7 48.8 39.9 | 52.2 49.9 47.3; 4096 x 14336 26.8 27.7 24.1 | 37.3 29.4
// 28.8; 6144 x 4096 15.9 15.4 14.8 | 21.6 17.3 18.1; 4096 x 4096 12.1 12.7 11.5 | 16.5 14.2 12.6;
// 16384 x 2048 16.6 17.1 15.5 | 20.6 19.2 16.5; 8192 x 28672 83 83 75 | 101 90 96.  Workgroups 128,
// 256, 512 at 8192 x 28672, 24 rows: 130, 90, 75; at 4096 x 14336 64, 128, 256, 512: 54, 33, 24, 27.
int few_rows(int M, int N, int K) {
  if (M > 64 || (M > 48 && K >= 8192 && (long)N * K > 80000000)) return 0;
  const int cols = N / 64, tiles = K / 64;
  int parts = 256 / cols;
  if (parts < 1) parts = 1;
  if (cols * parts < 192) parts = 512 / cols;
  if (tiles / parts > 128 && cols * parts <= 256) parts *= 2;
  if (parts > 8) parts = 8;
  if (parts > tiles / 6) parts = tiles / 6;
  if (parts < 1) parts = 1;
  const int depth = (tiles + parts - 1) / parts;
  return (tiles + depth - 1) / depth;
}

// The form and the parts of K (of six tiles at least) that the model gives the least time.  It
// picks what is 3 % slower than the best of all at the mean of the measured sizes, 1 % gated.
Plan plan_of(int M, int N, int K, bool gated) {
  if (gated && M <= 64) return Plan{kFew, 1, 0.0};
  if (const int parts = gated ? 0 : few_rows(M, N, K)) return Plan{kFew, parts, 0.0};
  Plan best{0, 1, 1e30};
  const double cols = gated ? 2.0 * N : N, w_mb = cols * K * 2e-6;
  for (int f = 0; f < 4; ++f) {
    const Form& form = kForms[f];
    if ((long)(gated ? 2 : 1) * N % form.bn) continue;
    const long blocks = (M + form.bm - 1) / form.bm * (long)(cols / form.bn);
    for (int parts = 1; parts <= 8; ++parts) {
      const int depth = (K / 64 + parts - 1) / parts;
      if (parts > 1 && (gated || depth < 6 || (K / 64 + depth - 1) / depth != parts ||
                        blocks * parts > 1024 || (double)parts * M * N > 64e6))
        continue;
      const long all = blocks * parts, round = 256 * form.pairs;
      const long full = all / round, rest = all % round;
      const bool alone = rest > 0 && rest <= 256;
      const double work =
          (alone ? form.own + depth * form.one : 0.0) +
          (full + (rest > 0 && !alone)) * (form.own + depth * form.two);
      const double read = w_mb * form.w_mb, w2 = work * work, r2 = read * read;
      const double us = form.start + sqrt(sqrt(w2 * w2 + r2 * r2)) +
                        (parts > 1 ? form.merge + form.merge_mb * parts * M * (double)N * 8e-6 : 0);
      if (us < best.us) best = Plan{f, parts, us};
    }
  }
  return best;
}

template <int BM, int BN, int SLOTS, int OCC, bool GATED, int HINT = 0>
void launch_form(__hip_bfloat16* y, float* part, const __hip_bfloat16* x, const __hip_bfloat16* w,
                 int M, int N, int K, int parts, hipStream_t stream) {
  const long blocks = (M + BM - 1) / BM * (long)(N / (GATED ? BN / 2 : BN));
  const int depth = (K / 64 + parts - 1) / parts * 64;
  hipLaunchKernelGGL((gemm_ring_kernel<BM, BN, SLOTS, OCC, GATED, HINT>),
                     dim3((blocks + 7) / 8 * 8, parts), dim3(256), 0, stream, y, part, x, w, M, N,
                     K, depth);
}

template <bool GATED>
void launch_plan(__hip_bfloat16* y, float* part, const __hip_bfloat16* x, const __hip_bfloat16* w,
                 int M, int N, int K, int plan, hipStream_t stream) {
  const int parts = plan & 15;
  switch (plan >> 4) {
    case 0: launch_form<256, 256, 4, 1, GATED>(y, part, x, w, M, N, K, parts, stream); break;
    case 1: launch_form<128, 256, 4, 1, GATED>(y, part, x, w, M, N, K, parts, stream); break;
    case 2: launch_form<128, 128, 4, 2, GATED>(y, part, x, w, M, N, K, parts, stream); break;
    case 3: launch_form<64, 128, 6, 2, GATED>(y, part, x, w, M, N, K, parts, stream); break;
    default:
      {
        // W that is read once and is large goes past the caches (24 rows: 28672 x 4096 46.4 ->
        // 39.9 us, 8192 x 3584 15.6 -> 13.8, 4096 x 4096 11.5 -> 11.5; 64 rows 12.6 -> 13.5)
        if (M <= 64 && (GATED ? 2L : 1L) * N * K >= 20000000)
          launch_form<64, 64, 8, 2, GATED, 2>(y, part, x, w, M, N, K, parts, stream);
        else
          launch_form<64, 64, 8, 2, GATED>(y, part, x, w, M, N, K, parts, stream);
      }
  }
}

// rows of W are found by 32 bits
bool fits(long M, long N, long K, bool gated) {
  return N % 128 == 0 && K % 64 == 0 && K > 0 && K < 1L << 23 && M > 0 && M < 1L << 24 &&
         N < 1L << 24 && (!gated || (N + 128) * K * 2 < 1L << 32);
}

}  // namespace

void launch_gemm_merge(__hip_bfloat16* y, const float* part, long plane, int parts, bool gated,
                       hipStream_t stream);

// Form and parts of a product: parts in the lowest four bits, each leaves M x N sums.
int gemm_ring_plan(int M, int N, int K, bool gated) {
  const Plan p = plan_of(M, N, K, gated);
  return p.form << 4 | p.parts;
}

// Whether a plan is one: a tile's columns fit, no part of K is empty.
bool gemm_ring_takes(int N, int K, int plan, bool gated) {
  const int form = plan >> 4, parts = plan & 15;
  if (plan < 0 || form > kFew || parts < 1 || parts > (gated ? 1 : 8)) return false;
  const int depth = (K / 64 + parts - 1) / parts;
  const int bn = form == kFew ? kForm4Cols : kForms[form].bn;
  return (gated ? 2L : 1L) * N % bn == 0 && (K / 64 + depth - 1) / depth == parts;
}

// Whether these tiles take a product from what would run it otherwise.  Time over that one's,
// cold weights, N x K: rows.
//  Against gemm_stream.hip's, 9 to 64 rows: 28672 x 4096 0.90 to 0.94; 4096 x 14336 0.77 to
//   0.90; 4096 x 4096 17 0.98, 64 0.76; 512 x 4096 0.96 to 0.66; 3072 x 2048 17 1.08, 40 0.95, 64
//   0.91; 2048 x 2048 32 1.12, 40 0.97.  2 | 12 rows: 28672 x 4096 0.99 | 0.94, 10240 x 8192 0.89 |
//   0.86, 2048 x 8192 0.96 | 0.94, 16384 x 2048 0.98 | 0.93, 4096 x 14336 1.02 | 0.97, 14336 x 4096
//   1.04 | 0.97; 6144 x 4096 1.13 | 1.10, 4096 x 7168 1.13 | 1.06, 8192 x 3584 1.07 | 1.03.
//  Against the library's:
//   65 to 256 rows: 4096 x 4096 0.60 to 0.99; 6144 x 4096 0.76 to 1.00; 4096 x 14336 0.82 to
//   0.97; 8192 x 8192 0.89 to 1.02; 2560 x 8192 0.54 to 0.90; 12288 and 14336 x 4096 and 8192
//   0.88 to 1.10, 28672 x 4096 0.99 to 1.14, 3072 x 2048 0.82 to 1.27, 1024 x 4096 1.11 to 1.25.
//   301 to 1024, long K: 4096 x 14336 0.81 to 0.97; 2048 x 8192 0.89 to 1.00; 8192 x 28672 0.63
//   to 1.12; others around 1: 4096 x 4096 0.97 to 1.16, 6144 x 4096 1.01 to 1.17.
//  Gated, against gemm_stream.hip's, 17 | 64 rows: 14336 x 4096 0.91 | 0.92, 6144 x 4096 0.86 |
//   0.82, 8192 x 2048 0.85 | 0.83, 7168 x 8192 1.01 | 0.79, 8192 x 8192 1.06 | 0.75, 11008 x 4096
//   1.07 | 0.80, 28672 x 8192 0.92 | 1.06; against the library's and its gate, where the model is below 0.92 of the library's
//   (fitted likewise): 8192 x 2048 0.78 to 0.93; 14336 x 4096 0.88 to 0.99 (768 rows: 1.07);
//   28672 x 8192 0.88 to 0.97 (256: 1.05); 4096 x 2048 0.54 to 0.94; 1024 x 2048 0.68 to 1.14.
bool gemm_ring_wins(long M, long N, long K, bool gated) {
  if (!fits(M, N, K, gated)) return false;
  if (gated) {
    if (M <= 64) {
      if (M <= 16 || N < 6144 || (M > 48 && N * K > 150000000)) return false;
      const long blocks = N / 32;   // one a CU, or nearly two
      return M > 32 || (blocks <= 256 ? K < 8192 : blocks >= 400);
    }
    if (N * K < 4000000) return false;
    const double tf = 4e-9 * M * N * K / 1.334;
    const double mb = (4e-6 * N * K + 2e-6 * M * (2.0 * N + K)) * 0.202;
    const double library = 12.9 + sqrt(tf * tf + mb * mb) + 0.6e-6 * M * N;
    return plan_of(M, N, K, true).us < 0.92 * library;
  }
  if (M <= 16) return M > 8 && (K >= 8192 ? N * K >= 16000000 : N * K >= 33000000);
  if (M <= 64)
    return N * K >= 2000000 && (K >= 4096 || N * K >= 16000000 || M >= 40);
  if (N * K < 6000000) return false;
  if (M <= 256) return K >= 3584 && N <= 10240;
  return M <= 1024 && 2 * K >= 7 * N;
}

// N % 128 == 0, K % 64 == 0, 0 < K < 2^23, x, W and y from 16-byte boundaries on
void launch_gemm_ring(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                      const __hip_bfloat16* w, int M, int N, int K, int plan, bool gated,
                      hipStream_t stream) {
  if (gated) launch_plan<true>(y, part, x, w, M, N, K, plan, stream);
  else launch_plan<false>(y, part, x, w, M, N, K, plan, stream);
  if ((plan & 15) > 1) launch_gemm_merge(y, part, (long)M * N, plan & 15, false, stream);
}

// the same, plain; parts of K are left as they are
void launch_gemm_ring_parts(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                            const __hip_bfloat16* w, int M, int N, int K, int plan,
                            hipStream_t stream) {
  launch_plan<false>(y, part, x, w, M, N, K, plan, stream);
}
