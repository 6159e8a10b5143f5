// Products of few rows with a whole weight matrix (decode, M <= 64):
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
//   1 row, 4 bits, the mean of the same four: 26.9 -> 10.9 (28672 x 4096: 18.3);
//   a llama-1b step of one stream 727 -> 486 us, a llama-3-8b one in 4 bits 1139 -> 753.

#include "common.h"

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;

namespace {

// QB: bits of a weight.  MT: 16-row tiles of x.  NT: 16-row tiles of W (of each half)
// of a wave.  WN x WK waves: along N (they share their tiles of x) and along K.
template <int QB, int MT, int NT, int WN, int WK, bool GATED>
__global__ __launch_bounds__(WN * WK * 64, 2) void gemm_stream_kernel(
    __hip_bfloat16* __restrict__ y,         // [M, N]
    float* __restrict__ part,               // [gridDim.y, GATED ? 2 : 1, M, N] (gridDim.y > 1)
    const __hip_bfloat16* __restrict__ x,   // [M, K]
    const void* __restrict__ w,             // [(GATED ? 2 : 1) * N, K]
    const float* __restrict__ scale,        // [N] (int8) | [N, K / 128] (4 bits)
    const int M, const int N, const int K) {
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
  const int n0 = (blockIdx.x * WN + wn) * (NT * 16);
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
  const __hip_bfloat16* x_at = x + (long)xr * K + xc * 8;

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
        t.x[p] = *reinterpret_cast<const u32x4_t*>(x_at + (long)first * K + i * KT);
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
        if constexpr (GATED) v = v / (1.f + __expf(-v)) * acc[NT + j][mt][r];
        y[(long)m * N + n] = __float2bfloat16(v);
      }
  }
}

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

// How a product is cut.  The lines are where they measured fastest (us, bf16 unless
// said; M = 1..16 | 23 | 61):
//   up to 16 rows of x, x is a small part of what is read and waves work alone:
//     4096 x 4096: WK 8 8.1, WK 4 9.5; 14336 x 4096 gated: WK 4 39.8, WK 8 42.0.
//   17..32: 14336 x 4096 gated: 2 x 2 43.4, 1 x 4 45.5; 4096 x 4096: 1 x 8 11.2, 4 x 2
//     over four workgroups and a merge 12.1; 4096 x 14336: the same two 27.4, 25.4.
//   33..64: every wave's own copy of x would cost more than W, 4 x 2 waves share it:
//     4096 x 14336: over four workgroups 34.9, 1 x 8 43.5; 14336 x 4096 gated: 2 x 2
//     48.4, 4 x 2 49.7; 28672 x 4096 int8: 4 x 2 42.8; 2048 x 2048: 1 x 8 9.4, 4 x 2 10.3.
enum class Cut { kWave8, kWave4, kShare22, kShare42 };

Cut cut_of(int M, int N, int K, bool gated) {
  if (M <= 16) return N / 16 < 512 ? Cut::kWave8 : Cut::kWave4;
  if (M <= 32) {
    if (N >= 8192) return Cut::kShare22;
    if (K >= 8192) return Cut::kShare42;
    return N / 16 < 320 ? Cut::kWave8 : Cut::kWave4;
  }
  if (K < 4096 && N < 8192) return Cut::kWave8;
  return gated ? Cut::kShare22 : Cut::kShare42;
}

template <int QB, int MT, bool GATED>
void launch_mt(__hip_bfloat16* y, float* part, const __hip_bfloat16* x, const void* w,
               const float* s, int M, int N, int K, int parts, hipStream_t stream) {
#define GO(WN, WK)                                                                            \
  hipLaunchKernelGGL((gemm_stream_kernel<QB, MT, 1, WN, WK, GATED>),                          \
                     dim3(N / (16 * WN), parts), dim3(64 * WN * WK), 0, stream, y, part, x, w, \
                     s, M, N, K)
  const Cut cut = cut_of(M, N, K, GATED);
  if constexpr (MT == 1) {
    if (cut == Cut::kWave8) GO(1, 8);
    else GO(1, 4);
  } else {
    switch (cut) {
      case Cut::kWave8: GO(1, 8); break;
      case Cut::kWave4: GO(1, 4); break;
      case Cut::kShare22: GO(2, 2); break;
      case Cut::kShare42:
        // the gated form takes this cut for few columns only
        GO(4, 2);
        break;
    }
  }
#undef GO
  if (parts > 1) {
    const long plane = (long)M * N;
    hipLaunchKernelGGL((gemm_stream_merge_kernel<GATED>), dim3((plane / 4 + 255) / 256),
                       dim3(256), 0, stream, y, part, plane, parts);
  }
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
// as many as make one a CU.  A function of shapes.
int gemm_stream_parts(int M, int N, int K, bool gated) {
  if (cut_of(M, N, K, gated) != Cut::kShare42) return 1;
  const int wgs = N / 64;
  int parts = (256 + wgs - 1) / wgs;
  if (parts > 8) parts = 8;
  const int most = K / 1024 > 0 ? K / 1024 : 1;   // four tiles of 128 a wave at least
  return parts < most ? parts : most;
}

// M <= 64, N % 64 == 0, K % 64 == 0 (rounded weights: K % 128 == 0)
void launch_gemm_stream(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                        const __hip_bfloat16* w, int M, int N, int K, int parts,
                        hipStream_t stream) {
  launch_q<16, false>(y, part, x, w, nullptr, M, N, K, parts, stream);
}

void launch_gemm_stream_gated(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                              const __hip_bfloat16* w13, int M, int I, int K, int parts,
                              hipStream_t stream) {
  launch_q<16, true>(y, part, x, w13, nullptr, M, I, K, parts, stream);
}

void launch_gemm_stream_q(__hip_bfloat16* y, float* part, const __hip_bfloat16* x,
                          const unsigned char* wq, const float* scale, int qbits, int M, int N,
                          int K, int parts, hipStream_t stream) {
  if (qbits == 8)
    launch_q<8, false>(y, part, x, wq, scale, M, N, K, parts, stream);
  else
    launch_q<4, false>(y, part, x, wq, scale, M, N, K, parts, stream);
}
