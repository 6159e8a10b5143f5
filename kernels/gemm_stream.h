// Kernel of the few-row products (described in gemm_stream.hip; moe_gemm.hip runs it
// per expert).
#pragma once

#include "common.h"
#include "moe_tiles.h"

namespace gemm_stream {

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;


// QB: bits of a weight.  MT: 16-row tiles of x.  NT: 16-row tiles of W (of each half)
// of a wave.  WN x WK waves: along N (they share their tiles of x) and along K.
// MODE: what becomes of the sums (kPlain ... of moe_tiles.h).  GROUPED: rows of x and y
// are sorted by expert, w holds one matrix per expert and blocks find their expert,
// columns and up to 16 MT rows of its segment by themselves.
template <int QB, int MT, int NT, int WN, int WK, int MODE, bool GROUPED = false>
__global__ __launch_bounds__(WN * WK * 64, 2) void gemm_stream_kernel(
    __hip_bfloat16* __restrict__ y,         // [M, N]
    float* __restrict__ part,               // [gridDim.y, GATED ? 2 : 1, M, N] (gridDim.y > 1)
    const __hip_bfloat16* __restrict__ x,   // [M, K]
    const void* __restrict__ w,             // [(GATED ? 2 : 1) * N, K]
    const float* __restrict__ scale,        // [N] (int8) | [N, K / 128] (4 bits)
    int M, const int N, const int K, const moe::Segments segs = moe::Segments{},
    const float limit = 0.f) {
  constexpr bool GATED = moe::gated(MODE);
  static_assert(!GROUPED || QB == 16, "experts' weights are bf16");
  constexpr int KT = QB != 4 && MT == 4 ? 64 : 128;    // inputs of a tile (4 bits: a group)
  constexpr bool DEEP = QB != 4 || MT < 4;             // two tiles on their way, or one
  constexpr int WT = GATED ? 2 * NT : NT;              // W tiles
  constexpr int WB = KT * QB / 8;                      // bytes of a W row in a tile
  constexpr int WL = WB / 16;                          // lanes (16-byte chunks) per W row
  constexpr int WP = WT * WL / 4;                      // load passes of W
  constexpr int XL = KT / 8;                           // lanes per x row
  constexpr int XP = MT * XL / 4;                      // load passes of x, by WN waves
  constexpr int XW = (XP + WN - 1) / WN;
  constexpr int W_BYTES = WT * 16 * WB, X_BYTES = MT * 16 * KT * 2;
  constexpr int STEPS = KT / 32;                       // matrix steps of a tile
  constexpr int WAVES = WN * WK;
  constexpr int XBUF = WN > 1 ? 2 : 1;     // shared tiles of x: one is read, one written
  constexpr int LDS = WAVES * W_BYTES + WK * XBUF * X_BYTES;
  static_assert(WK == 1 || LDS >= WAVES * WT * MT * 1024, "the waves' results fit");

  __shared__ __align__(16) char lds[LDS];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, quad = lane >> 4;
  const int wn = wave % WN, wk = wave / WN;
  int n_blk = blockIdx.x, row0 = 0;
  if constexpr (GROUPED) {
    const moe::Tile at = moe::find_tile(segs, 16 * MT, N / (16 * NT * WN));
    if (at.rows == 0) return;
    n_blk = at.n;
    M = at.rows;
    row0 = at.row0;
    y += (long)at.row0 * N;
    w = static_cast<const char*>(w) + (long)at.expert * (GATED ? 2 : 1) * N * K * 2;
  }
  const int n0 = (n_blk * WN + wn) * (NT * 16);
  char* w_lds = lds + wave * W_BYTES;
  char* x_lds = lds + WAVES * W_BYTES + wk * XBUF * X_BYTES;
  const long w_row_bytes = (long)K * QB / 8;
  const int tiles = (K + KT - 1) / KT;
  const int step = gridDim.y * WK;                     // K in turns over workgroups and waves

  // chunk c of row r lies at chunk c ^ swizzle(r): eight rows' equal chunks differ in
  // their banks
  auto swz_w = [](int r) { return WL == 16 ? r & 7 : WL == 8 ? (r >> 1) & 3 : (r >> 2) & 3; };
  auto swz_x = [](int r) { return XL == 16 ? r & 7 : (r >> 1) & 3; };
  // first W row of tile i
  auto w_row = [&](int i) { return i < NT ? n0 + i * 16 : N + n0 + (i - NT) * 16; };

  // where this lane's loads come from (pass p: rows p * 64 / lanes-per-row + ...)
  const int wr = lane / WL, wc = lane % WL;    // row within a pass, chunk
  const int xr = lane / XL, xc = lane % XL;
  const char* w_at[WP];
#pragma unroll
  for (int p = 0; p < WP; ++p) {
    const int r = p * (64 / WL) + wr;
    w_at[p] = static_cast<const char*>(w) + (w_row(r / 16) + r % 16) * w_row_bytes + wc * 16;
  }
  // (rows of x past M are not loaded)
  const __hip_bfloat16* x_at[XW];
#pragma unroll
  for (int p = 0; p < XW; ++p) {
    const int r = (p * WN + wn) * (64 / XL) + xr;
    long row = row0 + r;
    if constexpr (GROUPED) {
      if (segs.rows != nullptr && r < M) row = segs.rows[row];
    }
    x_at[p] = x + row * K + xc * 8;
  }

  struct Tile {
    u32x4_t w[WP], x[XW];
    float s[QB == 4 ? WT : 1];
  };
  auto load = [&](Tile& t, int i) {
    // the last tile of a K that is no multiple of KT: its missing half is zero
    const bool w_in = QB != 16 || i * KT + wc * 8 < K;
    const bool x_in = QB != 16 || i * KT + xc * 8 < K;
#pragma unroll
    for (int p = 0; p < WP; ++p) {
      t.w[p] = u32x4_t{};
      if (w_in)
        t.w[p] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4_t*>(w_at[p] + (long)i * WB));
    }
#pragma unroll
    for (int p = 0; p < XW; ++p) {
      const int first = (p * WN + wn) * (64 / XL);
      t.x[p] = u32x4_t{};
      if (first + xr < M && x_in)
        t.x[p] = *reinterpret_cast<const u32x4_t*>(x_at[p] + i * KT);
    }
    if constexpr (QB == 4) {
#pragma unroll
      for (int j = 0; j < WT; ++j) t.s[j] = 2.f * scale[(long)(w_row(j) + col) * (K / 128) + i];
    }
  };
  auto stage = [&](const Tile& t, char* xs) {
#pragma unroll
    for (int p = 0; p < WP; ++p) {
      const int r = p * (64 / WL) + wr;
      *reinterpret_cast<u32x4_t*>(w_lds + r * WB + (wc ^ swz_w(r)) * 16) = t.w[p];
    }
#pragma unroll
    for (int p = 0; p < XW; ++p) {
      const int r = (p * WN + wn) * (64 / XL) + xr;
      if (XP % WN != 0 && p * WN + wn >= XP) continue;
      u32x4_t v = t.x[p];
      if constexpr (QB == 4) {   // inputs 0 4 1 5 2 6 3 7, as the weights are unpacked
        const u32x4_t o = v;
        v[0] = __builtin_amdgcn_perm(o[2], o[0], 0x05040100);
        v[1] = __builtin_amdgcn_perm(o[2], o[0], 0x07060302);
        v[2] = __builtin_amdgcn_perm(o[3], o[1], 0x05040100);
        v[3] = __builtin_amdgcn_perm(o[3], o[1], 0x07060302);
      }
      *reinterpret_cast<u32x4_t*>(xs + r * KT * 2 + (xc ^ swz_x(r)) * 16) = v;
    }
    // other lanes of this wave read it: LDS keeps a wave's order, the compiler has to
    asm volatile("" ::: "memory");
  };
  const char* xs = x_lds;
  auto x_frag = [&](int mt, int chunk) {
    const int r = mt * 16 + col;
    return *reinterpret_cast<const bf16x8_t*>(xs + r * KT * 2 + (chunk ^ swz_x(r)) * 16);
  };
  auto w_chunk = [&](int i, int chunk) {
    const int r = i * 16 + col;
    return *reinterpret_cast<const u32x4_t*>(w_lds + r * WB + (chunk ^ swz_w(r)) * 16);
  };

  f32x4_t acc[WT][MT];
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[i][mt] = f32x4_t{};

  auto compute = [&](const float* s) {
    if constexpr (QB == 16) {
#pragma unroll
      for (int st = 0; st < STEPS; ++st) {
        bf16x8_t xf[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[mt] = x_frag(mt, st * 4 + quad);
#pragma unroll
        for (int i = 0; i < WT; ++i) {
          const bf16x8_t wf = __builtin_bit_cast(bf16x8_t, w_chunk(i, st * 4 + quad));
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[i][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt], wf, acc[i][mt], 0, 0, 0);
        }
      }
    } else if constexpr (QB == 8) {
      // a lane's 16-byte chunk holds inputs of two matrix steps
#pragma unroll
      for (int h = 0; h < STEPS / 2; ++h) {
        bf16x8_t xf[2][MT];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) xf[j][mt] = x_frag(mt, h * 8 + quad * 2 + j);
#pragma unroll
        for (int i = 0; i < WT; ++i) {
          const u32x4_t c = w_chunk(i, h * 4 + quad);
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            union { unsigned u[4]; bf16x8_t v; } wf;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
              const unsigned two = c[2 * j + d / 2] >> (d % 2 * 16);
              const float a = (float)(signed char)(two & 0xff);
              const float b = (float)(signed char)((two >> 8) & 0xff);
              // whole numbers of 8 bits: the upper half of the float is all of it
              wf.u[d] = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
              acc[i][mt] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[j][mt], wf.v, acc[i][mt], 0, 0, 0);
          }
        }
      }
    } else {
      // a lane's chunk holds inputs of all four steps; the tile is one group
      bf16x8_t off;
#pragma unroll
      for (int j = 0; j < 8; ++j) off[j] = (short)0xc140;   // -12
      u32x4_t c[WT];
      f32x4_t part[WT][MT], base[MT];
#pragma unroll
      for (int i = 0; i < WT; ++i) c[i] = w_chunk(i, quad);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        base[mt] = f32x4_t{};
#pragma unroll
        for (int i = 0; i < WT; ++i) part[i][mt] = f32x4_t{};
      }
#pragma unroll
      for (int st = 0; st < STEPS; ++st) {
        bf16x8_t xf[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          xf[mt] = x_frag(mt, quad * 4 + st);
          base[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt], off, base[mt], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < WT; ++i) {
          union { unsigned u[4]; bf16x8_t v; } wf;
#pragma unroll
          for (int d = 0; d < 4; ++d)
            wf.u[d] = ((d == 0 ? c[i][st] << 3 : c[i][st] >> (4 * d - 3)) & 0x00780078u) |
                      0x41004100u;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            part[i][mt] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mt], wf.v, part[i][mt], 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[i][mt][r] =
                __builtin_fmaf(s[i], part[i][mt][r] + base[mt][r], acc[i][mt][r]);
    }
    asm volatile("" ::: "memory");
  };

  // the next tiles are on their way while one is worked on; waves that share x keep
  // in step (one barrier a tile: the tile written next is not the one being read)
  Tile ta, tb;
  int buf = 0;
  auto turn = [&](Tile& t, int i, int next) {
    float s[QB == 4 ? WT : 1];
    char* to = x_lds + buf * X_BYTES;
    if (i < tiles) stage(t, to);
    if constexpr (QB == 4) {
#pragma unroll
      for (int j = 0; j < WT; ++j) s[j] = t.s[j];
    }
    if (next < tiles) load(t, next);
    if constexpr (WN > 1) {
      __syncthreads();
      buf ^= 1;
    }
    xs = to;
    if (i < tiles) compute(s);
  };
  const int first = blockIdx.y * WK;
  int i = first + wk;
  if (i < tiles) load(ta, i);
  if constexpr (DEEP) {
    if (i + step < tiles) load(tb, i + step);
    for (int at = first; at < tiles; at += 2 * step, i += 2 * step) {
      turn(ta, i, i + 2 * step);
      if (at + step < tiles) turn(tb, i + step, i + 3 * step);
    }
  } else {
    for (int at = first; at < tiles; at += step, i += step) turn(ta, i, i + step);
  }

  // ---- the sums of the waves along K become one --------------------------------
  if constexpr (WK > 1) {
    __syncthreads();
    f32x4_t* all = reinterpret_cast<f32x4_t*>(lds);
    if (wk > 0) {
#pragma unroll
      for (int j = 0; j < WT; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          all[((wave * WT + j) * MT + mt) * 64 + lane] = acc[j][mt];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int v = 1; v < WK; ++v)
#pragma unroll
      for (int j = 0; j < WT; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[j][mt] += all[(((v * WN + wn) * WT + j) * MT + mt) * 64 + lane];
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + j * 16 + col;
    float sa = 1.f;
    if constexpr (QB == 8) sa = scale[n];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = mt * 16 + quad * 4 + r;
        if (m >= M) continue;
        float v = acc[j][mt][r];
        if constexpr (QB == 8) v *= sa;
        if (gridDim.y > 1) {
          const long plane = (long)M * N, at = (long)m * N + n;
          part[blockIdx.y * (GATED ? 2 : 1) * plane + at] = v;
          if constexpr (GATED) part[(blockIdx.y * 2 + 1) * plane + at] = acc[NT + j][mt][r];
          continue;
        }
        v = moe::finish<MODE>(v, acc[GATED ? NT + j : j][mt][r], limit);
        y[(long)m * N + n] = __float2bfloat16(v);
      }
  }
}

}  // namespace gemm_stream
