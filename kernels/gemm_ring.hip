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
//   plain 512 x 4096 x 14336 84 -> 69; 65 x 4096 x 14336 37 -> 26; 192 x 4096 x 4096 33 -> 19;
//     128 x 6144 x 4096 26 -> 20; 128 x 8192 x 28672 113 -> 93
// What did not pay: tiles of 256 x 128 beside 128 x 256 (within 1 %), five slots of 128 x 128
// (2 % here and there), 64 x 256.

#include <algorithm>

#include "ring_gemm.h"
#include "lora_shrink.h"
#include "moe_tiles.h"

namespace {

using ring_gemm::f32x4_t;

// Tile `tile` of y, part `own` of K; part [parts, M, N] (parts > 1); depth: K of a part
template <int BM, int BN, int SLOTS, bool GATED, int HINT>
DEVINLINE void product(char* lds, __hip_bfloat16* __restrict__ y, float* __restrict__ part,
                       const __hip_bfloat16* __restrict__ x, const __hip_bfloat16* __restrict__ w,
                       const int M, const int N, const int K, const int depth, const int tile,
                       const int own, const int parts) {
  using R = ring_gemm::Ring<BM, BN, 2, 2, SLOTS, HINT>;
  constexpr int COLS = GATED ? BN / 2 : BN;              // outputs of a block
  constexpr int OUT = GATED ? R::kTN / 2 : R::kTN;       // output tiles of a wave
  // Each XCD has a run of neighbours: bands of up to eight tiles of rows, column by column,
  // so that the tiles that run at a time share rows of x and of W in its L2
  const int m_tiles = (M + BM - 1) / BM, n_tiles = N / COLS, blocks = m_tiles * n_tiles;
  const int per_xcd = (blocks + 7) / 8, slot = tile / 8;
  const int id = (tile % 8) * per_xcd + slot;
  if (slot >= per_xcd || id >= blocks) return;
  const int band = id / (8 * n_tiles), in = id % (8 * n_tiles), high = min(8, m_tiles - band * 8);
  const int m0 = (band * 8 + in % high) * BM, n0 = in / high * COLS, k0 = own * depth;

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
      if (!GATED && parts > 1) {
        float* to = part + own * ((long)M * N) + at + j * 16;
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

// grid (tiles of y, parts of K)
template <int BM, int BN, int SLOTS, int OCC, bool GATED, int HINT = 0>
__global__ __launch_bounds__(256, OCC) void gemm_ring_kernel(
    __hip_bfloat16* __restrict__ y, float* __restrict__ part,
    const __hip_bfloat16* __restrict__ x, const __hip_bfloat16* __restrict__ w, const int M,
    const int N, const int K, const int depth) {
  __shared__ __align__(16) char lds[ring_gemm::Ring<BM, BN, 2, 2, SLOTS, HINT>::kLds];
  product<BM, BN, SLOTS, GATED, HINT>(lds, y, part, x, w, M, N, K, depth, blockIdx.x, blockIdx.y,
                                      gridDim.y);
}

// The same, and beside it what the adapters of its rows need of x: `ahead` workgroups (a multiple of
// eight, so that tiles stay on their XCDs) that begin first, on CUs that the product's leave
// free or beside them.  In a launch of their own they took 4.0 to 5.2 us and a gap, all of it latency;
// here the product's weights go by meanwhile.  With expand, us, 61 rows, 4 adapters of rank 16, in two
// launches and in one: 6144 x 4096 24.6 20.0, 4096 x 4096 18.3 16.3, gated 28672 x 4096 66.9 63.2, 4096 x 14336
// 36.0 33.6; 24 rows 4096 x 4096 16.2 14.5, 32 rows 3072 x 2048 14.4 10.6.
constexpr int kShrinkTiles = 2;   // 16-wide tiles of a workgroup: one form for all ranks

template <int BM, int BN, int SLOTS, int OCC, int HINT>
__global__ __launch_bounds__(256, OCC) void gemm_ring_lora(
    __hip_bfloat16* __restrict__ y, float* __restrict__ part,
    const __hip_bfloat16* __restrict__ x, const __hip_bfloat16* __restrict__ w, const int M,
    const int N, const int K, const int depth, const int parts, const int tiles,
    const lora::Shrink shrink, const int adapters, const int ahead) {
  using R = ring_gemm::Ring<BM, BN, 2, 2, SLOTS, HINT>;
  static_assert(R::kLds >= lora::shrink_lds(kShrinkTiles) && lora::kShrinkWaves == 4, "shared");
  __shared__ __align__(16) char lds[R::kLds];
  int id = blockIdx.x;
  if (id < ahead) {
    const int wide = (shrink.PR + 16 * kShrinkTiles - 1) / (16 * kShrinkTiles);
    const int cut = id % shrink.cuts, row = id / shrink.cuts % wide;
    id /= shrink.cuts * wide;
    const int groups = lora::groups_of(lora::kWindow, adapters);   // of a window
    lora::shrink<kShrinkTiles, true>(shrink, cut, adapters, id / groups * lora::kWindow,
                                     id % groups, row * 16 * kShrinkTiles, lds);
    return;
  }
  id -= ahead;
  product<BM, BN, SLOTS, false, HINT>(lds, y, part, x, w, M, N, K, depth, id % tiles, id / tiles,
                                      parts);
}

// A tile's form and what its time is made of, in us, fitted to some 25000 measured products of 65
// to 4096 rows (50 shapes of W of the presets and their shards, weights from HBM; standard
// deviation 6 %), then moved a little towards the better choices: the start; a workgroup's start
// and end and its tiles of 64 inputs, alone on its CU and in pairs, less a share for rows that
// do not exist; the reading of W, more with every further tile of rows up to five; and a second
// launch for parts of K.  The share of empty rows and `again` are of the whole.
struct Form {
  int bm, bn, pairs;
  double start, own, one, two, merge, merge_mb, merge_part, w_mb, again, empty;
};
constexpr Form kForms[] = {
    {256, 256, 1, 0.14, 12.0, 1.07, 1.07, 2.3, 0.125, 1.10, 0.186, 0.52, 0.0},
    {128, 256, 1, 0.20, 5.4, 0.77, 0.77, 4.9, 0.120, 0.55, 0.170, 0.31, 0.39},
    {128, 128, 2, 2.46, 2.0, 0.53, 0.97, 2.8, 0.142, 0.26, 0.167, 0.36, 0.30},
    {64, 128, 2, 3.00, 0.4, 0.38, 0.74, 3.1, 0.154, 0.16, 0.180, 0.23, 0.60},
    {64, 64, 2, 2.83, 0.5, 0.27, 0.53, 2.1, 0.202, 0.14, 0.205, 0.07, 0.60},
};
constexpr int kNarrow = 3, kFew = 4, kFormCount = 5;   // 64 x 128, 64 x 64

struct Plan {
  int form, parts;
  double us;
};

// parts of K without an empty one
int even_parts(int K, int parts) {
  const int depth = (K / 64 + parts - 1) / parts;
  return (K / 64 + depth - 1) / depth;
}

// Up to 64 rows x is one tile and W comes by once: workgroups of 64 rows of W, as many as there
// are CUs (K cut), or two a CU where that leaves a quarter of them idle or K stays long, and W
// past the caches.  us, the streaming kernel | 64 x 128 by a cost model | here, N x K, 24 |
// 64 rows: 28672 x 4096 44.7 48.8 39.9 | 52.2 49.9 47.3; 4096 x 14336 26.8 27.7 24.1 | 37.3 29.4
// 28.8; 4096 x 4096 12.1 12.7 11.5 | 16.5 14.2 12.6; 16384 x 2048 16.6 17.1 15.5 | 20.6 19.2 16.5.
// Workgroups 128, 256, 512 of 64 columns at 8192 x 28672, 24 rows: 130, 90, 75; at 4096 x 14336 64, 128,
// 256, 512: 54, 33, 24, 27; 172 and 344 at 11008 x 4096: 20.2, 24.2.
// Short K is cut less, eight tiles a part: 40 rows, 3072 x 2048 in 4 8.9 (in 5 9.4, whole 10.7), 8192
// x 1024 whole 7.3 (in 2 8.0).  Past 48 rows of very many weights the tile of 128 columns reads x half
// as often, 128 | 64 columns: 64 rows, 57344 x 8192 175 | 183, 8192 x 28672 in 4 90 | 96 (14336 x 8192
// 60 | 47, 28672 x 8192 98 | 89).
// For fewer rows too it is faster where columns of 64 would be cut and still be two a CU (one a CU then),
// and, with K cut further, where they would be cut in two (half the barriers for as many bytes).  us, 64 |
// 128 columns, 17 rows, 64 rows: 10240 x 8192 in 3 32.2 | 30.5, 38.7 | 33.7; 10240 x 2048 in 3 12.6 | 11.8,
// 17.4 | 15.8; 14336 x 14336 in 2 75.9 | 63.3, 94.2 | 72.6; 9, 24, 48 rows, 8192 x 28672 in 4 72.2 | 71.2, 76.2 |
// 72.6, 87.2 | 77.4; 5120 x 28672 in 6 49.3 | 48.0, 52.3 | 49.3, 60.7 | 52.3; 10240 x 28672 in 3 97 | 91, 104 |
// 93, 118 | 97; of 23 such matrices, 9 to 64 rows, none is 1 % slower; in 2 | in 4: 6144 x 4096 13.7 | 12.7, 17.2 | 16.7;
// 8192 x 4096 16.5 | 14.6, 18.2 | 16.4; 6144 x 14336 33.1 | 31.5, 43.4 | 38.5; but 6144 x 2048 8.9 | 9.6;
// in 2 | in 3: 8192 x 8192 27.3 | 25.1, 29.8 | 28.7; but 6144 x 8192 22.2 | 22.8, 27.5 | 28.0.
Plan few_rows(int M, int N, int K) {
  const int cols = N / 64, tiles = K / 64;
  int parts = 256 / cols;
  if (parts < 1) parts = 1;
  if (cols * parts < 192 && 512 / cols > 2) parts = 512 / cols;
  if (tiles / parts > 128 && cols * parts <= 256) parts *= 2;
  if (parts > 8) parts = 8;
  const int most = tiles < 32 ? 1 : tiles < 64 ? tiles / 8 : tiles / 6;
  if (parts > most) parts = most;
  if (parts < 1) parts = 1;
  bool wide = (M > 48 && K >= 8192 && (K >= 16384 || (long)N * K > 400000000)) ||
              (parts > 1 && cols * parts > 256);
  if (parts == 2 && cols <= 128 && K >= 4096) {
    const int more = K <= 6144 || K >= 12288 ? 4 : cols >= 120 ? 3 : 2;
    wide = wide || more > 2;
    parts = more;
  }
  return Plan{wide && N % 128 == 0 ? kNarrow : kFew, even_parts(K, parts), 0.0};
}

// The form and the parts of K (of six tiles at least) that the model gives the least time.  It
// picks what is 0.5 % slower than the best of all at the mean of the measured sizes, 6 % at one in
// a hundred.  A cut tile's workgroups go where blockIdx.x does, eight XCDs of 32 CUs in turn:
// rounds are counted there (84 tiles in three parts are 33 workgroups on some XCDs, two rounds,
// though all are 252: 1.5 times the time of 80 tiles).
Plan plan_of(int M, int N, int K, bool gated) {
  // (gated: past one and a half rounds of two a CU of 64 rows of W, which are two then, 128 are one.  us, 64 |
  // 128 at 17, 40, 64 rows, up to the line and past it: 24576 x 2048 36.7 | 39.9, 37.3 | 41.1, 39.7 | 42.8, 24704
  // x 2048 43.4 | 40.6, 44.5 | 42.0, 48.1 | 43.5; 24576 x 4096 63 | 70, 66 | 73, 71 | 76, 24704 x 4096 75 | 71, 79 |
  // 74, 87 | 78; 24576 x 5120 80 | 88, 90 | 93, 99 | 100, 24704 x 5120 96 | 87, 109 | 93, 122 | 100; farther off,
  // 20480 x 5120 76 | 84, 94 | 96, 28672 x 8192 146 | 142, 155 | 145, 174 | 152)
  if (M <= 64) return gated ? Plan{N > 24576 ? kNarrow : kFew, 1, 0.0} : few_rows(M, N, K);
  Plan best{0, 1, 1e30};
  const double cols = gated ? 2.0 * N : N, w_mb = cols * K * 2e-6;
  for (int f = 0; f < kFormCount; ++f) {
    const Form& form = kForms[f];
    if ((long)(gated ? 2 : 1) * N % form.bn) continue;
    const long m_tiles = (M + form.bm - 1) / form.bm, blocks = m_tiles * (long)(cols / form.bn);
    const double full_rows = 1.0 - form.empty * (1.0 - (double)M / (m_tiles * form.bm));
    const double read =
        w_mb * form.w_mb * (1.0 + form.again * (m_tiles > 5 ? 4 : m_tiles - 1));
    for (int parts = 1; parts <= 8; ++parts) {
      const int depth = (K / 64 + parts - 1) / parts;
      if (parts > 1 && (gated || depth < 6 || even_parts(K, parts) != parts ||
                        blocks * parts > 1400 || (double)parts * M * N > 64e6))
        continue;
      const long all = (blocks + 7) / 8 * parts, round = 32 * form.pairs;   // of an XCD
      const long full = all / round, rest = all % round;
      const bool alone = rest > 0 && rest <= 32;
      const double work = full_rows * ((alone ? form.own + depth * form.one : 0.0) +
                                       (full + (rest > 0 && !alone)) *
                                           (form.own + depth * form.two));
      const double w2 = work * work, r2 = read * read;
      const double us =
          form.start + sqrt(sqrt(w2 * w2 + r2 * r2)) +
          (parts > 1 ? form.merge + form.merge_mb * parts * M * (double)N * 8e-6 +
                           form.merge_part * (parts - 2)
                     : 0);
      if (us < best.us) best = Plan{f, parts, us};
    }
  }
  return best;
}

// W that is read once and is large goes past the caches, by tiles of up to 64 rows from 20 million weights
// on, by larger ones from 40 (64 x 64, 24 rows: 28672 x 4096 46.4 -> 39.9 us, 8192 x 3584 15.6 -> 13.8, 4096 x
// 4096 11.5 -> 11.5, 64 rows 12.6 -> 13.5; 64 x 128, 17, 40, 64 rows: 8192 x 4096 17.3 -> 14.6, 17.8 -> 15.4, 18.7 ->
// 16.4, 6144 x 4096 13.6 -> 13.0, 15.8 -> 14.8, 17.2 -> 16.9, 5120 x 4096 12.6 -> 12.0, 13.8 -> 13.7, 15.1 -> 15.5,
// 3072 x 8192 18.4 -> 17.6, 21.4 -> 19.4, 22.5 -> 21.3, but 10240 x 2048 12.6 -> 12.2, 13.8 -> 14.1, 14.8 -> 16.1,
// and below the line 4096 x 4096 11.7 -> 11.4, 13.0 -> 12.8, 14.2 -> 14.5; larger tiles, all rows in one: 8192
// x 8192 by 128 x 128 0.88 of the time, 4096 x 14336 0.91, 5120 x 8192 0.97, but 7168 x 4096 1.02, 6144 x
// 4096 1.05)
bool read_once(int M, long weights, int form) {
  return M <= kForms[form].bm && weights >= (form >= kNarrow ? 20000000 : 40000000);
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

// The workgroups that shrink M rows beside a product
int beside(int M, int PR, int adapters, int cuts) {
  const int wide = (PR + 16 * kShrinkTiles - 1) / (16 * kShrinkTiles);
  const int groups = M / lora::kWindow * lora::groups_of(lora::kWindow, adapters) +
                     lora::groups_of(M % lora::kWindow, adapters);
  return (cuts * wide * groups + 7) / 8 * 8;
}

template <int BM, int BN, int SLOTS, int OCC, int HINT>
void launch_lora_form(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                      const __hip_bfloat16* w, int M, int N, int K, int parts,
                      const lora::Shrink& shrink, int adapters, hipStream_t stream) {
  const long tiles = ((M + BM - 1) / BM * (long)(N / BN) + 7) / 8 * 8;
  const int ahead = beside(M, shrink.PR, adapters, shrink.cuts);
  const int depth = (K / 64 + parts - 1) / parts * 64;
  hipLaunchKernelGGL((gemm_ring_lora<BM, BN, SLOTS, OCC, HINT>), dim3(ahead + tiles * parts),
                     dim3(256), 0, stream, y, part, x, w, M, N, K, depth, parts, (int)tiles, shrink,
                     adapters, ahead);
}

template <bool GATED>
void launch_plan(__hip_bfloat16* y, float* part, const __hip_bfloat16* x, const __hip_bfloat16* w,
                 int M, int N, int K, int plan, hipStream_t stream) {
  const int parts = plan & 15, form = plan >> 4;
  const bool once = read_once(M, (GATED ? 2L : 1L) * N * K, form);
#define GO(BM, BN, SLOTS, OCC)                                                         \
  if (once) launch_form<BM, BN, SLOTS, OCC, GATED, 2>(y, part, x, w, M, N, K, parts, stream); \
  else launch_form<BM, BN, SLOTS, OCC, GATED>(y, part, x, w, M, N, K, parts, stream); \
  break
  switch (form) {
    case 0: GO(256, 256, 4, 1);
    case 1: GO(128, 256, 4, 1);
    case 2: GO(128, 128, 4, 2);
    case 3: GO(64, 128, 6, 2);
    default: GO(64, 64, 8, 2);
  }
#undef GO
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

// Whether a product's weights go past the caches.
bool gemm_ring_reads_once(int M, int N, int K, int plan, bool gated) {
  return read_once(M, (gated ? 2L : 1L) * N * K, plan >> 4);
}

// Whether a plan is one: a tile's columns fit, no part of K is empty.
bool gemm_ring_takes(int N, int K, int plan, bool gated) {
  const int form = plan >> 4, parts = plan & 15;
  if (plan < 0 || form >= kFormCount || parts < 1 || parts > (gated ? 1 : 8)) return false;
  return (gated ? 2L : 1L) * N % kForms[form].bn == 0 && even_parts(K, parts) == parts;
}

// Rows of a plain product past 64 that the tiles take because K is so long, and tiles of 128 x
// 128 so few, that K can be cut over three workgroups and more.  Time over the library's, weights
// from HBM, N x K: first and last row of the rule, and the one past it:
//   1280 x 8192: 257 0.73, 700 0.84; 2048 x 8192: 129 0.65, 700 0.83; 2560 x 8192: 224 0.73, 512
//   0.86, 513 0.85; 4096 x 14336: 65 0.58, 640 0.77, 700 0.86; 5120 x 8192: 65 0.82, 512 0.81, 513
//   1.06; 7168 x 8192: 65 0.87, 384 0.94, 448 0.87; 8192 x 8192: 65 0.87, 256 0.69, 340 1.12; 8192 x
//   14336: 65 0.69, 256 0.59, 340 0.92; 10240 x 8192: 65 0.45, 256 0.65, 257 1.02.
// (7168 x 8192, 301 to 384 rows, are 4 to 10 % slower than eight-wave tiles with two whole tiles of
// K in LDS were there.)
bool gemm_block_takes(long M, long N, long K) {
  if (K < 8192 || N > 12288 || N < 128) return false;
  if (N < 2048) return M >= 257 && M <= 700;
  if (N < 2560) return M >= 129 && M <= 700;
  if (N < 3072) return M >= 200 && M <= 512;
  const long last = 168 / (N / 128) * 128;
  return M >= 65 && M <= (last < 700 ? last : 700);
}

// Whether these tiles take a product from what would run it otherwise.  Time over that one's,
// weights from HBM, N x K: rows.
//  Against gemm_stream.hip's, 9 to 64 rows: 28672 x 4096 0.94 to 0.92; 4096 x 14336 12 1.03, 17
//   0.93, 64 0.79; 4096 x 4096 17 1.04, 32 0.97, 64 0.82; 2048 x 4096 17 1.06, 32 1.0, 64 0.85; 8192 x
//   2048 17 0.83; 16384 x 2048 12 0.83; 10240 x 8192 12 0.83, 64 0.96; 14336 x 8192 0.90 to 0.85; 8192
//   x 28672 0.89 to 0.91.  Left there: 12 rows of 6144 x 4096 1.05, 8192 x 4096 1.05 to 1.12 (half of
//   the CUs without a tile, or K cut), 8192 x 3584 1.08; short K, 40 | 64 rows: 4096 x 1024 1.08 |
//   1.05, 4096 x 1792 1.15 | 1.13, 2048 x 1024 1.15 | 1.13, where 8192 x 1024 has 0.74 | 0.69 and
//   4864 x 896 0.88 | 0.87 (past 4096 columns the streaming workgroups are more than CUs).
//   (Taken with K of 2048: 3072 x 2048 1.06 | 1.02, 4096 x 2048 1.06 | 1.04.)
//  Against the library's, plain:
//   65 to 256 rows, K from 3584 on: 4096 x 4096 0.58 to 0.95; 6144 x 4096 0.64 to 0.93; 4096 x 14336
//   0.41 to 0.78; 8192 x 4096 0.75 to 1.01; 2048 x 4096 0.84 to 0.96; 14336 x 4096 0.90 to 1.04.
//   257 to 1024, long K: 4096 x 14336 0.64 to 0.86; 2048 x 8192 0.74 to 0.91; 1280 x 8192 0.71 to
//   0.89; 8192 x 28672 0.59 to 1.00, 513 to 768 rows 0.99 to 1.09, 900 0.96, 1024 0.93; others around 1: 4096 x 4096 0.91 to
//   1.17, 6144 x 4096 0.92 to 1.13.
//  Gated, against gemm_stream.hip's, 17 | 64 rows: 14336 x 4096 0.91 | 0.92, 6144 x 4096 0.86 |
//   0.82, 8192 x 2048 0.85 | 0.83, 7168 x 8192 1.01 | 0.79, 8192 x 8192 1.06 | 0.75, 11008 x 4096
//   1.07 | 0.80, 28672 x 8192 0.89 | 0.94.
//  Gated, past 64 rows, against the library's product (or the plain one by these tiles, where they
//   take it) and its gate: where the model is below 1.05 of a model of the library's fitted likewise
//   (14 %), below 0.98 for tiles of 256 x 256, whose last round costs most, and below 0.9 of its own
//   for the plain one.  8192 x 2048 0.78 to 0.93; 14336 x 4096 0.88 to 0.99 (340 rows: 1.04); 28672
//   x 8192 0.80 to 0.99; 4096 x 2048 0.54 to 1.00; 2048 x 2048 0.55 to 0.94.
bool gemm_ring_wins(long M, long N, long K, bool gated) {
  if (!fits(M, N, K, gated)) return false;
  if (gated) {
    if (M <= 64) {
      if (M <= 16 || N < 6144 || (M > 48 && N * K > 150000000 && N <= 24576)) return false;
      const long blocks = N / 32;   // one a CU, or nearly two
      return M > 32 || (blocks <= 256 ? K < 8192 : blocks >= 400);
    }
    if (N * K < 4000000) return false;
    const Plan plan = plan_of(M, N, K, true);
    if (gemm_block_takes(M, 2 * N, K) || gemm_ring_wins(M, 2 * N, K, false))
      return plan.us < 0.9 * (plan_of(M, 2 * N, K, false).us + 2.5 + 1.2e-6 * M * N);
    const double products = 4e-9 * M * N * K / 1.294;
    const double bytes = 4e-6 * N * K * 0.179 + 2e-6 * M * (2.0 * N + K) * 0.39;
    const double library = 12.9 + sqrt(products * products + bytes * bytes);
    return plan.us < (plan.form == 0 ? 0.98 : 1.05) * library;
  }
  if (M <= 16) return M > 8 && (K >= 8192 ? N * K >= 16000000 : N * K >= 33000000 && N >= 12288);
  if (M <= 64) {
    if (K >= 4096 || N * K >= 16000000) return N * K >= 2000000;
    return M >= 40 && (N > 4096 ? N * K >= 2000000 : K >= 2048 && N * K >= 6000000);
  }
  if (N * K < 6000000) return false;
  if (M <= 256) return K >= 3584 && N <= 10240;
  return M <= 1024 && 2 * K >= 7 * N && (N * K <= 100000000 || M <= 512 || M > 832);
}

// Both questions of a plain product past 64 rows: 1 gemm_block_takes, 2 gemm_ring_wins, 0 neither
int gemm_tiles_route(long M, long N, long K) {
  if (M <= 64) return 0;
  return gemm_block_takes(M, N, K) ? 1 : gemm_ring_wins(M, N, K, false) ? 2 : 0;
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

// Parts of K for the adapters' shrink beside a product by `plan`, 0: in a launch of its own.  There
// is time beside a product, so K is cut less than it is alone and expand has fewer sums to add, but
// a wave's eight steps are short of the shortest product (K 8192, 40 rows, rank 64: four parts 22.1 us,
// eight 18.9, alone 21.4).  Each of its workgroups holds the LDS of one of the product's, two a CU:
// up to one a CU they are done when the product's later ones would begin; more keep it waiting
// (sides: alone, beside; 4096 x 14336, 96 rows, 32 adapters of rank 8: 481 workgroups 38.9 52.9; 4096 x
// 4096, 512 rows, 8 of rank 64: 384 70.9 83.6; but 256 rows, 2 of rank 64: 144 42.6 40.3).
int gemm_ring_lora_cuts(int M, int K, int L, int PR, int plan) {
  const int cuts = std::min(lora_shrink_cuts(M, K), std::max(4, K / 1024));
  return plan >> 4 >= 2 && beside(M, PR, L, cuts) <= 256 ? cuts : 0;
}

// Whether these tiles take a product that has adapters, whatever takes it without them: beside other
// products the shrink is a launch of its own, the deltas go over their rounded results, and where K is
// cut the sum of the parts is one more; here it is two launches, three where the shrink has no room beside
// the product (gemm_ring_lora_cuts: many adapters or tokens, high ranks).  Of the adapters the rule sees their
// rank, for one row of many columns.  us with the deltas, otherwise | here, 4 adapters of rank 16 (captured, cold weights), N x K: rows
//   up to 16 rows: 6144 x 4096 2 19.2 | 15.8, 16 21.7 | 16.8; 28672 x 4096 gated 2 49.7 | 45.3; 4096 x 14336
//    8 30.5 | 26.6; 2048 x 2048 12 11.3 | 8.8; 57344 x 8192 gated 2 174 | 163; 768 x 768 2 8.8 | 9.0; not
//    4096 x 1792 12.3 | 13.7 (too short to be cut, 64 workgroups); of one row 6144 x 4096 16.4 | 15.0, 2048
//    x 2048 9.3 | 7.8, but 4096 x 4096 12.5 | 13.3, 57344 x 8192 153 | 161; of one row and rank 8, whose
//    expand is little, gated 16384 x 2048 18.8 | 19.5, 28672 x 4096 45.9 | 47.5, 7168 x 4096 16.9 | 15.7;
//   17 to 128: 2048 x 2048 64 16.2 | 9.2; 3072 x 2048 32 15.1 | 10.1, 65 20.7 | 12.7; 16384 x 2048 gated
//    128 35.5 | 32.2; 28672 x 4096 gated 80 81.8 | 62.7, 128 73.2 | 65.9, 160 76.4 | 82.8; 57344 x 8192
//    gated 65 207 | 172;
//   up to 256: 3072 x 2048 24.3 | 19.4; 16384 x 2048 gated 44.7 | 38.5; 57344 x 8192 gated 269 | 234;
//   up to 512: 4096 x 4096 301 37.8 | 33.3, 512 43.0 | 40.4; 2048 x 2048 512 22.3 | 16.9; 10240 x 8192 400
//    110 | 100; 1536 x 4096 301 26.8 | 20.5; 3072 x 2048 400 28.1 | 28.5, 512 29.6 | 32.4; 6144 x 4096
//    400 50.5 | 55.4; 16384 x 2048 gated 301 46.8 | 48.8.
// (Of other ranks and numbers of adapters: as far or further apart but for rank 64 at 400 to 512 rows,
// 0.98 to 1.03 of the others.)
bool gemm_ring_lora_wins(long M, long N, long K, int rank) {
  if (!fits(M, N, K, false)) return false;
  if (M <= 64 ? gemm_ring_wins(M, N, K, false) : gemm_tiles_route(M, N, K) != 0) return true;
  const long size = N * K;
  if (M == 1)
    return size <= 6000000 || (size <= 300000000 && (K >= 8192 || (N > 4096 && (rank > 8 || N < 16384))));
  if (M <= 16) return K <= 1024 || K >= 2048 || N > 4096;
  if (M <= 128) return true;
  if (M <= 256) return size <= 34000000 || K >= 8192;
  if (M > 512) return false;
  return (K >= 8192 && size <= 100000000) ||
         size <= (M <= 320 || K >= 4096 ? 17000000 : 5000000);
}

// launch_gemm_ring_parts and, in the same launch, tmp [cuts, M, PR] = the rows of A x of each
// row's adapter, in parts
void launch_gemm_ring_lora(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                           const __hip_bfloat16* w, int M, int N, int K, int plan, float* tmp,
                           const __hip_bfloat16* a, const int* slots, int L, int PR, int cuts,
                           hipStream_t stream) {
  const int parts = plan & 15, form = plan >> 4;
  const lora::Shrink shrink{tmp, x, a, slots, M, PR, K, cuts};
  const bool once = read_once(M, (long)N * K, form);
#define GO(BM, BN, SLOTS, OCC)                                                              \
  if (once) launch_lora_form<BM, BN, SLOTS, OCC, 2>(y, part, x, w, M, N, K, parts, shrink, L, stream); \
  else launch_lora_form<BM, BN, SLOTS, OCC, 0>(y, part, x, w, M, N, K, parts, shrink, L, stream); \
  break
  switch (form) {
    case 2: GO(128, 128, 4, 2);
    case 3: GO(64, 128, 6, 2);
    default: GO(64, 64, 8, 2);
  }
#undef GO
}
