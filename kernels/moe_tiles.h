// What the products over experts' segments share: where a block's rows and columns lie,
// and what becomes of a sum.
#pragma once

#include "common.h"

namespace moe {

// plain | silu(g) u | relu(v)^2 | the clamped gate of common.h
enum Mode { kPlain = 0, kSilu = 1, kRelu2 = 2, kClamped = 3 };

constexpr bool gated(int mode) { return mode == kSilu || mode == kClamped; }

template <int MODE> DEVINLINE float finish(float v, float u, float limit) {
  if constexpr (MODE == kClamped) return clamped_gate(v, u, limit);
  if constexpr (MODE == kSilu) return v / (1.f + __expf(-v)) * u;
  if constexpr (MODE == kRelu2) {
    v = fmaxf(v, 0.f);
    return v * v;
  }
  return v;
}

struct Segments {
  const int* off;    // [experts + 1] first row of each expert's segment, device
  int experts;
  const int* rows;   // row of x that each sorted row is, or null: x is sorted itself
};

struct Tile {
  int expert, n, row0, rows;   // rows == 0: nothing to do
};

// Blocks are numbered expert by expert, columns by columns, row chunks of at most
// `chunk` rows innermost, and the numbers are dealt out so that each of the eight XCDs
// (blockIdx.x % 8) has a run of neighbours: chunks that read the same columns of W, and
// columns that read the same rows, meet in one L2.  Segment sizes stay on the device;
// the launch covers the most blocks there can be (max_blocks) and the rest end here.
DEVINLINE int count_chunks(const Segments& s, int chunk) {   // of all experts
  const int lane = threadIdx.x & 63;
  int total = 0;
  for (int e0 = 0; e0 < s.experts; e0 += 64) {
    const int e = e0 + lane;
    int c = 0;
    if (e < s.experts) c = (s.off[e + 1] - s.off[e] + chunk - 1) / chunk;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) c += __shfl_xor(c, d, 64);
    total += c;
  }
  return __builtin_amdgcn_readfirstlane(total);
}

// The tile of number `id`, which is one of count_chunks(s, chunk) * n_tiles
DEVINLINE Tile tile_of(const Segments& s, int chunk, int n_tiles, int id) {
  const int lane = threadIdx.x & 63;
  for (int e0 = 0; e0 < s.experts; e0 += 64) {
    const int e = e0 + lane;
    int lo = 0, rows = 0;
    if (e < s.experts) {
      lo = s.off[e];
      rows = s.off[e + 1] - lo;
    }
    const int c = (rows + chunk - 1) / chunk;
    int upto = c;   // chunks of experts e0 .. e
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(upto, d, 64);
      if (lane >= d) upto += v;
    }
    const int all = __builtin_amdgcn_readfirstlane(__shfl(upto, 63, 64)) * n_tiles;
    if (id >= all) {
      id -= all;
      continue;
    }
    // the first expert whose blocks reach past id
    const int at = __builtin_amdgcn_readfirstlane(__popcll(__ballot(upto * n_tiles <= id)));
    const int ce = __builtin_amdgcn_readfirstlane(__shfl(c, at, 64));
    const int before = __builtin_amdgcn_readfirstlane(__shfl(upto, at, 64)) - ce;
    const int local = id - before * n_tiles;
    const int n = local / ce, m = local % ce;
    const int lo_e = __builtin_amdgcn_readfirstlane(__shfl(lo, at, 64));
    const int rows_e = __builtin_amdgcn_readfirstlane(__shfl(rows, at, 64));
    return Tile{e0 + at, n, lo_e + m * chunk, min(chunk, rows_e - m * chunk)};
  }
  return Tile{0, 0, 0, 0};
}

DEVINLINE Tile find_tile(const Segments& s, int chunk, int n_tiles) {
  const int blocks = count_chunks(s, chunk) * n_tiles, per_xcd = (blocks + 7) / 8;
  const int slot = blockIdx.x / 8, id = (blockIdx.x % 8) * per_xcd + slot;
  if (slot >= per_xcd || id >= blocks) return Tile{0, 0, 0, 0};
  return tile_of(s, chunk, n_tiles, id);
}

// The most blocks that rows of these many experts can make, a multiple of eight.
inline long max_blocks(long rows, int experts, int chunk, int n_tiles) {
  const long filled = rows < experts ? rows : experts;   // segments that are not empty
  return ((rows / chunk + filled) * n_tiles + 7) / 8 * 8;
}

}  // namespace moe
