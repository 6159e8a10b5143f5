// Products of one row with a weight matrix (one stream):
//   y[n] = sum_k x[k] W[n, k],  or  silu(x Wg^T) * (x Wu^T) for W = [Wg; Wu],
// W in bf16 or in 4 bits (offset 8, a scale per row and 128 inputs).
//
// Bound by the bytes of W.  With a single row the tiles of gemm_stream.h spend their time on
// instructions, not on bytes: 15 of 16 rows of their x tiles are empty, and are loaded,
// turned and staged for every 1 KB of 4-bit weights.  Here x is put into LDS once a
// workgroup, in the order that a lane's weights leave their words; a wave takes four rows
// of W at a time (two of each half when gated), a lane 16 bytes of each, and multiplies
// pairs by
// v_dot2_f32_bf16 into f32.  4-bit weights enter as 8 + n / 2, -12 times the sum of x
// takes the offset out, the doubled scale goes onto the f32 sum of a lane's 32 inputs.
//
// us over 1.5 GB of weights in turn, gemm_stream.h -> here (at 6.2 TB/s; reads in sequence
// reach 6.4), N x K:
//   4 bits: 28672 x 4096 23.7 -> 18.1 (10.1), 6144 x 4096 8.9 -> 7.2 (2.2), 4096 x 4096 6.7 ->
//     5.8 (1.4), 4096 x 14336 17.4 -> 13.6 (5.0);
//   bf16: 14336 x 4096 gated 41.7 -> 36.9 (37.9), 8192 x 2048 gated 15.7 -> 13.4 (10.8), 2048 x
//     8192 11.4 -> 8.9 (5.4), 2048 x 2048 5.1 -> 4.2 (1.4), 32000 x 2048 27.8 -> 22.8 (21.1);
//   a llama-1b step 486 -> 433 us, a llama-3-8b one in 4 bits 751 -> 638.
// With two rows the same way is no faster (28672 x 4096 23.7, bf16 4096 x 4096 9.9 against
// 8.8), in int8 it is slower with one (28672 x 4096 26 against 25).

#include "common.h"
#include "moe_tiles.h"

namespace {

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf2_t;

constexpr int kRows = 4;    // of W, a wave
constexpr int kWaves = 4;

DEVINLINE float dot2(unsigned a, unsigned b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2_t, a),
                                         __builtin_bit_cast(bf2_t, b), c, false);
}

// KS: waves that K is dealt to, the others take other rows of W.
template <int QB, bool GATED, int KS>
__global__ __launch_bounds__(64 * kWaves) void gemm_row_kernel(
    __hip_bfloat16* __restrict__ y,         // [N]
    const __hip_bfloat16* __restrict__ x,   // [K]
    const unsigned char* __restrict__ w,    // [(GATED ? 2 : 1) * N, K]
    const float* __restrict__ scale,        // [N, K / 128] (4 bits)
    const int N, const int K) {
  constexpr int PER = 128 / QB;             // weights of a lane's 16 bytes
  constexpr int CPL = PER / 8;              // 16-byte chunks of x that go with them
  constexpr int SEG = 64 * PER;             // inputs of a wave's load
  constexpr int OUT = GATED ? kRows / 2 : kRows, RS = kWaves / KS, COLS = RS * OUT;
  extern __shared__ __align__(16) char lds[];   // x [segments, CPL, 64] chunks
  __shared__ float sums[2][kWaves][kRows];

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ks = wave % KS, rs = wave / KS;
  const int segs = (K + SEG - 1) / SEG, blocks = N / COLS;
  const long row_bytes = (long)K * QB / 8;
  const unsigned char* at[kRows];
  const float* s_at[QB == 4 ? kRows : 1];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const int n = rs * OUT + (GATED && r >= OUT ? N + r - OUT : r);
    at[r] = w + n * row_bytes + lane * 16;
    if constexpr (QB == 4) s_at[r] = scale + (long)n * (K / 128) + lane / 4;
  }
  u32x4_t ahead[kRows];
  float s_ahead[QB == 4 ? kRows : 1];
  auto load = [&](int block, int seg) {
    const bool in = seg * SEG + lane * PER < K;   // K is a multiple of a lane's share
    const long rows = (long)block * COLS;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      ahead[r] = u32x4_t{};
      if (in)
        ahead[r] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4_t*>(at[r] + rows * row_bytes + (long)seg * 1024));
      if constexpr (QB == 4)
        s_ahead[r] = in ? 2.f * s_at[r][rows * (K / 128) + seg * (SEG / 128)] : 0.f;
    }
  };
  if (ks < segs) load(blockIdx.x, ks);

  const int chunks = segs * 64 * CPL;       // of x, past K zero
  u32x4_t* xs = reinterpret_cast<u32x4_t*>(lds);
  for (int c = threadIdx.x; c < chunks; c += 64 * kWaves) {
    u32x4_t v{};
    if (c * 8 < K) v = *reinterpret_cast<const u32x4_t*>(x + c * 8);
    if constexpr (QB == 4) {   // inputs 0 4 1 5 2 6 3 7, as the weights are unpacked
      const u32x4_t o = v;
      v[0] = __builtin_amdgcn_perm(o[2], o[0], 0x05040100);
      v[1] = __builtin_amdgcn_perm(o[2], o[0], 0x07060302);
      v[2] = __builtin_amdgcn_perm(o[3], o[1], 0x05040100);
      v[3] = __builtin_amdgcn_perm(o[3], o[1], 0x07060302);
    }
    const int in = c % (64 * CPL);
    xs[c - in + in % CPL * 64 + in / CPL] = v;
  }
  __syncthreads();

  int turn = 0;
  for (int block = blockIdx.x; block < blocks; block += gridDim.x, turn ^= 1) {
    float acc[kRows] = {};
    for (int seg = ks; seg < segs; seg += KS) {
      u32x4_t q[kRows];
      float s[QB == 4 ? kRows : 1];
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        q[r] = ahead[r];
        if constexpr (QB == 4) s[r] = s_ahead[r];
      }
      if (seg + KS < segs) load(block, seg + KS);
      else if (block + gridDim.x < blocks) load(block + gridDim.x, ks);
      float part[kRows] = {}, base = 0.f;
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        const u32x4_t xv = xs[(seg * CPL + j) * 64 + lane];
        if constexpr (QB == 4) {
#pragma unroll
          for (int d = 0; d < 4; ++d) base = dot2(xv[d], 0xc140c140u, base);   // -12
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            unsigned two;
            if constexpr (QB == 16) {
              two = q[r][d];
            } else {   // 8 + n / 2
              two =
                  ((d == 0 ? q[r][j] << 3 : q[r][j] >> (4 * d - 3)) & 0x00780078u) | 0x41004100u;
            }
            float& to = QB == 4 ? part[r] : acc[r];
            to = dot2(xv[d], two, to);
          }
      }
      if constexpr (QB == 4) {
#pragma unroll
        for (int r = 0; r < kRows; ++r) acc[r] = __builtin_fmaf(s[r], part[r] + base, acc[r]);
      }
    }

    // four rows' sums over 64 lanes in one: row lane / 32 + 2 (lane / 16 % 2)
    const bool up = lane & 32, odd = lane & 16;
    const float a = (up ? acc[1] : acc[0]) + __shfl_xor(up ? acc[0] : acc[1], 32, 64);
    const float b = (up ? acc[3] : acc[2]) + __shfl_xor(up ? acc[2] : acc[3], 32, 64);
    float v = (odd ? b : a) + __shfl_xor(odd ? a : b, 16, 64);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane % 16 == 0) sums[turn][wave][lane / 32 + 2 * (lane / 16 % 2)] = v;
    __syncthreads();   // the next turn writes elsewhere
    if (threadIdx.x < COLS) {
      const int o = threadIdx.x % OUT, first = threadIdx.x / OUT * KS;
      const int n = block * COLS + threadIdx.x;
      float g = 0.f, u = 0.f;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        g += sums[turn][first + k][o];
        if constexpr (GATED) u += sums[turn][first + k][OUT + o];
      }
      y[n] = __float2bfloat16(moe::finish<GATED ? moe::kSilu : moe::kPlain>(g, u, 0.f));
    }
  }
}

template <int QB, bool GATED, int KS>
void launch(__hip_bfloat16* y, const __hip_bfloat16* x, const void* w, const float* scale, int N,
            int K, hipStream_t stream) {
  constexpr int SEG = 64 * 128 / QB, COLS = kWaves / KS * (GATED ? kRows / 2 : kRows);
  static_assert(128 % COLS == 0, "whole workgroups");
  // four workgroups a CU walk the rows (28672 x 4096 4 bits: 17.0 us, two 19.1, all 19.2)
  const int blocks = N / COLS;
  hipLaunchKernelGGL((gemm_row_kernel<QB, GATED, KS>), dim3(blocks < 1024 ? blocks : 1024),
                     dim3(64 * kWaves), (K + SEG - 1) / SEG * SEG * 2, stream, y, x,
                     static_cast<const unsigned char*>(w), scale, N, K);
}

}  // namespace

// x is kept in LDS
bool gemm_row_fits(int qbits, int K) { return qbits != 8 && K <= 28672; }

// N % 128 == 0, K % 64 == 0 (4 bits: K % 128 == 0).  K is dealt to all four waves in bf16
// (2048 x 8192 8.8 us, to two 10.0, to one 14.2); in 4 bits a load covers 2048 inputs, and
// rows go first where they are many (28672 x 4096: one 17.0, two 21.7; 2048 x 8192: four
// 6.0, two 7.0, one 9.9).
void launch_gemm_row(__hip_bfloat16* y, const __hip_bfloat16* x, const void* w,
                     const float* scale, int qbits, int N, int K, bool gated,
                     hipStream_t stream) {
  if (qbits == 16) {
    if (gated) launch<16, true, 4>(y, x, w, scale, N, K, stream);
    else launch<16, false, 4>(y, x, w, scale, N, K, stream);
  } else if (K > 2048 * 3 && N <= 8192) {
    launch<4, false, 4>(y, x, w, scale, N, K, stream);
  } else if (K > 2048 && N <= 16384) {
    launch<4, false, 2>(y, x, w, scale, N, K, stream);
  } else {
    launch<4, false, 1>(y, x, w, scale, N, K, stream);
  }
}
