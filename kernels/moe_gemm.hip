// Grouped products over experts' segments: one launch covers every
// expert's rows of the batch sorted by expert,
//
//   h[r, :]  = silu(x[r]·Wg_e^T) * (x[r]·Wu_e^T)   (gated, w13 = [E, 2I, H])
//   y[r, :]  = h[r]·W2_e^T                          (plain, w2  = [E, H, I])
//   a[r, :]  = relu(x[r]·Wu_e^T)^2                  (squared relu, w = [E, I, H])
//   h[r, :]  = clamped gate of x[r]·Wg_e^T, x[r]·Wu_e^T (see common.h; as gated)
//
// where e = the expert owning sorted row r (seg_off[e] <= r < seg_off[e+1]).  Counts
// never leave the GPU: blocks find their expert, rows and columns (moe_tiles.h).  The
// sorted rows need not exist: with a list of rows (x_rows) row r is x[x_rows[r]].
//
// Few rows an expert: bound by the bytes of W, the streaming kernel of gemm_stream.h.
// More: ring_gemm.h's tiles of 128 x 128 to 256 x 256; the gated form takes half of a tile's
// columns from each half of W, arranged so that a wave holds the gate and the up sum of the
// same output.
//
// Measured, 8 experts of 14336 x 4096 (two experts a token, MI355X): a layer's three
// products and its routing, 33 tokens 723 -> 452 us (4.7 -> 6.2 TB/s), 2949 tokens 1950 (eight
// waves on 256 x 256) -> 1670 us (1.25 PFLOP/s; of the second product's 384 tiles, one and a half
// rounds of 256 CUs, the last 128 have K cut in two; with 400, 144 are left, which stay whole).

#include <algorithm>

#include "gemm_stream.h"
#include "ring_gemm.h"

namespace {

using ring_gemm::f32x4_t;

// Tiles that do not fill a last round of the chip leave CUs idle for as long as a whole one: 400
// tiles of 256 x 256 are 1.6 rounds of 256 CUs.  So K of the tiles behind the last whole round is
// cut in parts, a workgroup each, and the launch behind adds them up.
constexpr int kCus = 256;
constexpr int kMostParts = 2 * kCus - 1;   // of all those tiles

// A row's results are not to depend on its place among its expert's rows, which callers leave to
// the order of atomics: where the line falls between the chunks of an expert's rows in one column
// tile, the ones ahead of it are sums of the same parts too, made by one workgroup one after the other.
struct Rounds {
  int whole;          // tiles of one workgroup each
  int summed;         // tiles from here on are sums of parts
  int parts, depth;   // of these: parts of K, steps of a part
};

// A step takes 0.95 us where a workgroup has the chip's caches to itself and 1.5 beside 255 others
// (the smaller tiles are hardly faster: 128 x 256 stay whole), a part 0.22 us to store and to add, the
// launch 8.  4096 x 14336, 8 experts, tiles: whole tiles | with parts, us: 288 578 | 456, 384 620 | 578,
// 576 899 | 790; 16 experts, 6144 x 8192: 792 744 | 685.  432, whose last 176 tiles are left whole: 650 | 652.
// (Equal shares of all steps instead, whatever tile they belong to: 384 610 | 560, but 432
// 622 | 710: workgroups at different inputs find nothing of each other's in the caches.)
// Two launches decide alike, so the times are whole numbers, of 1 / 25600 us: there are ties (8192
// inputs, 120 tiles).
// shared: tiles ahead of the line whose chunks are of the same expert and column tile as one behind it
__host__ __device__ inline Rounds rounds_of(int tiles, int steps, int shared) {
  const int rest = tiles % kCus;
  Rounds best{tiles, tiles, 1, steps};
  if (rest == 0) return best;
  auto round = [](int blocks) { return blocks > 0 ? 24320L + 55 * blocks : 0; };   // a step of all
  long least = steps * round(rest);
  for (int parts = 2; parts <= 8 && parts * (rest + shared) <= kMostParts && parts * 8 <= steps;
       ++parts) {
    const int depth = ((steps + parts - 1) / parts + 1) / 2 * 2, blocks = rest * parts;
    const long time =
        depth * (round(blocks < kCus ? blocks : kCus) + round(blocks - kCus)) + 204800 + blocks * 5632;
    if (time < least) {
      least = time;
      best = Rounds{tiles - rest, tiles - rest - shared, parts, depth};
    }
  }
  return best;
}

DEVINLINE Rounds rounds_of(const moe::Segments& segs, int chunk, int n_tiles, int tiles, int steps) {
  const int line = tiles - tiles % kCus;
  if (line == tiles) return rounds_of(tiles, steps, 0);
  const moe::Tile at = moe::tile_of(segs, chunk, n_tiles, line);
  return rounds_of(tiles, steps, (at.row0 - segs.off[at.expert]) / chunk);
}

// What a lane holds of a tile: row i * 16 + lane % 16 of its wave's, columns in eights
template <typename R, int OUT, int MODE>
DEVINLINE void store(__hip_bfloat16* y, const moe::Tile& at, int N, int n0, int i,
                     const f32x4_t (&acc)[R::kTN], float limit) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / 2, wn = wave % 2, m = (wm * R::kTM + i) * 16 + (lane & 15);
  if (m >= at.rows) return;
  __hip_bfloat16* to = y + (long)(at.row0 + m) * N + n0 + wn * OUT * 16 + lane / 16 * 8;
#pragma unroll
  for (int j = 0; j < OUT; j += 2) {
    union { __hip_bfloat16 h[8]; uint4 u; } o;
#pragma unroll
    for (int r = 0; r < 8; ++r)
      o.h[r] = __float2bfloat16(moe::finish<MODE>(
          acc[j + r / 4][r % 4], acc[(moe::gated(MODE) ? OUT : 0) + j + r / 4][r % 4], limit));
    *reinterpret_cast<uint4*>(to + j * 16) = o.u;
  }
}

// part: null, or room for the parts that moe_gemm_scratch counts
template <int BM, int BN, int SLOTS, int OCC, int MODE>
__global__ __launch_bounds__(256, OCC) void moe_ring_kernel(
    __hip_bfloat16* __restrict__ y,        // [T, N]
    const __hip_bfloat16* __restrict__ x,  // [T, K] sorted by expert, or what segs.rows lists
    const __hip_bfloat16* __restrict__ w,  // [E, (gated ? 2 N : N), K]
    f32x4_t* __restrict__ part, const moe::Segments segs, const int N, const int K,
    const float limit) {
  using R = ring_gemm::Ring<BM, BN, 2, 2, SLOTS>;
  constexpr bool GATED = moe::gated(MODE), PARTED = !GATED && BM == 256;
  constexpr int COLS = GATED ? BN / 2 : BN;              // outputs of a block
  constexpr int OUT = GATED ? R::kTN / 2 : R::kTN;       // output tiles of a wave
  __shared__ __align__(16) char lds[R::kLds];

  const int steps = K / ring_gemm::kDepth, n_tiles = N / COLS;
  const int tiles = moe::count_chunks(segs, BM) * n_tiles;
  Rounds rounds{tiles, tiles, 1, steps};
  if (PARTED && part != nullptr) rounds = rounds_of(segs, BM, n_tiles, tiles, steps);
  const int per_xcd = (rounds.whole + 7) / 8, xcd = blockIdx.x % 8;
  const int slot = blockIdx.x / 8 - per_xcd;
  int id = xcd * per_xcd + blockIdx.x / 8, own = 0, end = 1;   // parts of K
  if (slot < 0) {
    if (id >= rounds.whole) return;
    if (id >= rounds.summed) end = rounds.parts;
  } else {   // part by part, so that what is read at a time is of the same inputs
    if constexpr (!PARTED) return;
    const int rest = tiles - rounds.whole, per = (rest * rounds.parts + 7) / 8;
    const int piece = xcd * per + slot;
    if (slot >= per || piece >= rest * rounds.parts) return;
    id = rounds.whole + piece % rest;
    own = piece / rest;
    end = own + 1;
  }
  const bool summed = PARTED && id >= rounds.summed;
  const moe::Tile at = moe::tile_of(segs, BM, n_tiles, id);
  const int n0 = at.n * COLS;
  const unsigned row_bytes = K * 2;
  f32x4_t acc[R::kTM][R::kTN];
  for (;;) {
    const int first = own * rounds.depth, k0 = first * ring_gemm::kDepth;
    R::clear(acc);
    R::run(acc, lds, reinterpret_cast<const char*>(x + k0),
           reinterpret_cast<const char*>(w + ((long)at.expert * (GATED ? 2 : 1) * N + n0) * K + k0),
           (summed ? min(rounds.depth, steps - first) : steps) * ring_gemm::kDepth,
           // rows past the segment: its last one, whose results are not written
           [&](int r) {
             const int row = at.row0 + min(r, at.rows - 1);
             return (segs.rows != nullptr ? segs.rows[row] : row) * row_bytes;
           },
           [&](int r) {   // a wave's output tiles of gates, then of the other half
             const int wave = r / (R::kTN * 16), in = r % (R::kTN * 16);
             const int half = in / (OUT * 16);
             return (half * N + wave * (OUT * 16) + R::out_col(in % (OUT * 16))) * row_bytes;
           });
    if (!summed) break;
    f32x4_t* to = part +
                  ((long)own * (tiles - rounds.summed) + id - rounds.summed) * (BM * BN / 4) +
                  threadIdx.x;
#pragma unroll
    for (int i = 0; i < R::kTM; ++i)
#pragma unroll
      for (int j = 0; j < R::kTN; ++j) to[(i * R::kTN + j) * 256] = acc[i][j];
    if (++own == end) return;
    block_gemm::meet();   // all have read what LDS holds
  }
#pragma unroll
  for (int i = 0; i < R::kTM; ++i) store<R, OUT, MODE>(y, at, N, n0, i, acc[i], limit);
}

// The parts of a tile become its results.  Grid (any, sixteenths of half of a tile's rows)
template <int BM, int BN, int MODE>
__global__ __launch_bounds__(256) void moe_parts_kernel(
    __hip_bfloat16* __restrict__ y, const f32x4_t* __restrict__ part, const moe::Segments segs,
    const int N, const int K, const float limit) {
  using R = ring_gemm::Ring<BM, BN, 2, 2, 4>;
  const int n_tiles = N / BN, i = blockIdx.y;
  const int tiles = moe::count_chunks(segs, BM) * n_tiles;
  const Rounds rounds = rounds_of(segs, BM, n_tiles, tiles, K / ring_gemm::kDepth);
  const int rest = tiles - rounds.summed;
  for (int own = blockIdx.x; own < rest; own += gridDim.x) {
    const moe::Tile at = moe::tile_of(segs, BM, n_tiles, rounds.summed + own);
    if (i * 16 >= at.rows) continue;   // (of the first half of its rows)
    f32x4_t acc[R::kTN];
#pragma unroll
    for (int j = 0; j < R::kTN; ++j) acc[j] = f32x4_t{};
    for (int p = 0; p < rounds.parts; ++p) {
      const f32x4_t* from =
          part + (long)(p * rest + own) * (BM * BN / 4) + i * (R::kTN * 256) + threadIdx.x;
#pragma unroll
      for (int j = 0; j < R::kTN; ++j) acc[j] += from[j * 256];
    }
    store<R, R::kTN, MODE>(y, at, N, at.n * BN, i, acc, limit);
  }
}

}  // namespace

// Which tile the products of more than some 52 rows an expert take: 0 256 x 256, 1 128 x 256, 2
// 128 x 128 (rows x columns of W), by the mean of the rows and, since a tile that runs alone on
// its CU takes as long as a full round of them, by how many tiles there are: us, 256 x 256 | 128 x 256
// | 128 x 128, experts x between (in), rows an expert, evenly spread, tiles of 256 x 256:
//   gated: 8 x 1792 (4096), 125, 112: 72 | 44 | 55; 4 x 512 (1024), 160, 16: 25 | 15 | 11; 8 x 3584
//   (4096), 160, 224: 117 | 129 | 140 (unevenly, 200: 173 | 135 | 153); 8 x 7168 (4096), 448, 200: 204 |
//   251 | 268.  About 240 rows some experts have more than 256, and one round of tiles becomes two:
//   8 x 3584 (4096), 249: 189 | 140 | 159, 16 x 2048 (2048), 249: 98 | 99 | 91.
//   plain: 8 of 4096 (14336), 222, 128: 298 | 235 | 281 (unevenly 294 | 402 | 369), 249, 256: 299 | 418
//   | 390; 8 of 4096 (3584), 222, 128: 65 | 49 | 53; 16 of 2048 (2048), 222, 128: 43 | 31 | 33; 4 of 1024
//   (512), 160, 16: 16 | 10 | 8; 16 of 4096 (3584), 222, 256: 107 | 133 | 145.
//   Short K (evenly, unevenly), where two tiles of 128 x 128 share a CU for less: 32 of 2048 (1024),
//   118: 34 | 37 | 31, 35 | 40 | 33; 245: 56 | 56 | 47, 59 | 55 | 48; 280: 66 | 59 | 56, 60 | 59 | 55;
//   420: 67 | 78 | 73, 86 | 76 | 72; 64 of 2048 (768), 140: 57 | 67 | 61, 55 | 63 | 55, 180: 58 | 72 |
//   66, 74 | 71 | 64 (256 x 256 are one tile an expert there, but two of the experts with more);
//   48 of 2048 (768), 280: 80 | 75 | 66, 75 | 78 | 66; 16 of 2048 (2048), whose 128 x 256 are one
//   round, 118: 44 | 28 | 35, 44 | 29 | 36, 245: 50 | 53 | 48, 51 | 55 | 48.
int moe_tile(int mean, int experts, long columns, int K, bool gated) {
  if (columns % 256 != 0) return 2;
  auto tiles = [&](long mean, long rows) {
    return (mean + rows - 1) / rows * experts * (columns / 256);
  };
  if (gated) {
    const long large = tiles(mean, 256);
    if (mean > (K >= 4096 ? 110 : 150) && large >= 192 && (large > 256 || mean <= 236 || mean > 256))
      return 0;
    return mean > 52 && K >= 4096 ? 1 : 2;
  }
  // some experts have more rows than the mean: from 228 on they are counted as two tiles
  const long more = mean * 9L / 8;
  if (mean > (K <= 2048 ? 300 : 220) && tiles(more, 256) >= 192) return 0;
  if (K <= 2048 && tiles(more, 128) > 256) return 2;
  return mean > 110 && tiles(mean, 128) >= 128 ? 1 : 2;
}

namespace {

template <int MODE>
void launch_mode(__hip_bfloat16* y, const __hip_bfloat16* x, const __hip_bfloat16* w,
                 const int* seg_off, const int* x_rows, int E, int N, int K, int T,
                 float limit, float* scratch, hipStream_t stream) {
  const moe::Segments segs{seg_off, E, x_rows};
  f32x4_t* part = reinterpret_cast<f32x4_t*>(scratch);
  const int cols = moe::gated(MODE) ? 2 : 1;
#define STREAM(MT, WN, WK)                                                                    \
  hipLaunchKernelGGL((gemm_stream::gemm_stream_kernel<16, MT, 1, WN, WK, MODE, true>),        \
                     dim3(moe::max_blocks(T, E, 16 * MT, N / (16 * WN))), dim3(64 * WN * WK), \
                     0, stream, y, nullptr, x, w, nullptr, 0, N, K, segs, limit)
#define TILES(BM, BN, SLOTS, OCC)                                                             \
  hipLaunchKernelGGL((moe_ring_kernel<BM, BN, SLOTS, OCC, MODE>),                             \
                     dim3(moe::max_blocks(T, E, BM, N * cols / BN) + (part ? kMostParts + 1 : 0)), \
                     dim3(256), 0, stream, y, x, w, part, segs, N, K, limit)
  // Rows an expert, us gated / plain of what is chosen and its neighbour (8 experts, 4096 in
  // and 14336 between; rows are spread at random):
  //    8: <1,1,4> 270, <1,2,2> 144 (<2,2,2> 271, <4,4,2> 143);
  //   17: <2,2,2> 278, <4,4,2> 144 (<4,4,2> 301, <2,2,2> 170);  25: <4,4,2> 305, 156
  //       (<2,2,2> 316, 197);  52: <4,4,2> 335, 171 (128 x 128 333, 166).
  // Tiles, 128 x 128 | 128 x 256 | 256 x 256, * is chosen:
  //   56: 327* 336* - / 163* 215 -;  100: 347 345* 387 / 179* 235 248;  125: 421 395 403* / 295
  //       244* 253;  200: 543 464 412* / 269 234* 285;  249: 629 591 505* / 391 426 311*;
  //   400: 908 836 705* / 505 429 331*.
  // and with 16 experts, 2048 in and between, where 128 x 256 are too few:
  //   64: 59* 66 - / 33* 37 -;  125: 69* 79 74 / 42 41* 46;  200: 89 81 78* / 43 42* 50.
  // (The eight-wave tiles before these took, gated / plain, 64: 357 / 227, 200: 529 / 269.)
  // Which of the tiles, and where they are too few for the chip: moe_tile below.
  //
  // That is with even loads.  The streaming form's workgroups, a chunk of 64 rows an expert and
  // two a CU, fill whole rounds at usual widths, and a few experts with more rows start another
  // round: plain products that are brim-full go to the large tiles earlier, where these fill
  // the chip or K is short.  16 experts of 4096 out and 3584 between, 128 tokens (mean 32) even |
  // by rank^-0.6: <4,4,2> 83 | 112, 128 x 128 85 | 85; 2048 and 2048: 33 | 47, 37 | 36; 8 of
  // 4096 and 3584, 128 x 128 at one workgroup a CU: <4,4,2> 46 | 49, 66 | 66.
  const int mean = T / E;
  // what the tiles do not take: rows of a block are found by 32 bits, results are stored by 16
  // bytes (the streaming form stores them one by one)
  const bool far = (long)N * cols * K * 2 >= 1L << 32 || (long)T * K * 2 >= 1L << 32 ||
                   reinterpret_cast<uintptr_t>(y) % 16 != 0;
  const long one = (long)E * (N / 64), last = one % 512;   // streaming workgroups
  const bool brim = !moe::gated(MODE) && (last == 0 || last > 460) &&
                    (K <= 2048 || (one >= 1024 && K <= 8192));
  if (mean <= 9 && moe::gated(MODE)) STREAM(1, 1, 4);
  else if (mean <= 9) STREAM(1, 2, 2);
  else if (mean <= 18 && moe::gated(MODE)) STREAM(2, 2, 2);
  else if (far || (mean <= 52 && !brim)) STREAM(4, 4, 2);
  else switch (moe_tile(mean, E, N * cols, K, moe::gated(MODE))) {
    case 0:
      TILES(256, 256, 4, 1);
      if constexpr (!moe::gated(MODE))
        if (part)
          hipLaunchKernelGGL((moe_parts_kernel<256, 256, MODE>), dim3(kCus / 2, 8), dim3(256), 0,
                             stream, y, part, segs, N, K, limit);
      break;
    case 1: TILES(128, 256, 4, 1); break;
    default: TILES(128, 128, 5, 2);
  }
#undef STREAM
#undef TILES
}

}  // namespace

// Floats of scratch that launch_moe_gemm wants, 0: none, whatever the segments hold.  From 8192 inputs
// on: below, parts save no more than they cost (7168, 416 tiles 323 | 330 us) and the launch that finds
// nothing to add is 2 to 4 us.  The segments' chunks of rows, at most T / 256 and one an expert, are not
// known here, so it is the most that any number of them wants: 8 experts of 14336 x 4096, 2949 tokens 87 MiB.
long moe_gemm_scratch(int E, int N, int K, int T, int mode) {
  if (mode == 1 || K < 8192 || T / E <= 52 || moe_tile(T / E, E, N, K, false) != 0) return 0;
  const int n_tiles = N / 256, most = T / 256 + std::min(T, E);
  const int shared = (long)most * n_tiles > kCus ? (T + 255) / 256 - 1 : 0;
  int pieces = 0;
  for (int chunks = 1; chunks <= std::min(most, kCus); ++chunks) {   // (what is left of a round repeats)
    const int rest = chunks * n_tiles % kCus;
    const Rounds rounds = rounds_of(rest, K / ring_gemm::kDepth, 0);
    // (chunks that share a line make no more parts of it)
    if (rounds.parts > 1)
      pieces = std::max(pieces, std::min(kMostParts, rounds.parts * (rest + shared)));
  }
  return pieces * (256L * 256);
}

void launch_moe_gemm(__hip_bfloat16* y, const __hip_bfloat16* x, const __hip_bfloat16* w,
                     const int* seg_off, const int* x_rows, int E, int N, int K, int T,
                     int mode, float* scratch, hipStream_t stream) {
  if (mode == 1)
    launch_mode<moe::kSilu>(y, x, w, seg_off, x_rows, E, N, K, T, 0.f, scratch, stream);
  else if (mode == 2)
    launch_mode<moe::kRelu2>(y, x, w, seg_off, x_rows, E, N, K, T, 0.f, scratch, stream);
  else
    launch_mode<moe::kPlain>(y, x, w, seg_off, x_rows, E, N, K, T, 0.f, scratch, stream);
}

void launch_moe_gemm_clamped(__hip_bfloat16* y, const __hip_bfloat16* x,
                             const __hip_bfloat16* w, const int* seg_off, int E, int N, int K,
                             int T, float limit, hipStream_t stream) {
  launch_mode<moe::kClamped>(y, x, w, seg_off, nullptr, E, N, K, T, limit, nullptr, stream);
}
