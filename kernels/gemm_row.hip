// Products of one row with a weight matrix (one stream):
//   y[n] = sum_k x[k] W[n, k],  or  silu(x Wg^T) * (x Wu^T) for W = [Wg; Wu],
// W in bf16, in int8 (a scale per row) or in 4 bits (offset 8, a scale per row and 128
// inputs), and what a layer does around them in the same launch: the norm ahead of a product,
// the rotation and the cache write behind the one for queries, keys and values.
//
// Bound by the bytes of W, small ones by the 1.9 us that a launch after another takes.  With
// a single row the tiles of gemm_stream.h spend their time on
// instructions, not on bytes: 15 of 16 rows of their x tiles are empty, and are loaded,
// turned and staged for every 1 KB of 4-bit weights.  Here x is put into LDS once a
// workgroup, in the order that a lane's weights leave their words; a wave takes four rows
// of W at a time (two of each half when gated), a lane 16 bytes of each, and multiplies
// pairs by
// v_dot2_f32_bf16 into f32.  int8 weights enter as whole numbers, 4-bit ones as 8 + n / 2:
// -12 times the sum of x takes the offset out, the doubled scale goes onto the f32 sums.
// Unpacking takes about as long as the bytes in 4 bits (three instructions a pair).
//
// us over 1 GB of weights in turn, gemm_stream.h -> here (at 6.2 TB/s; reads in sequence
// reach 6.4), N x K:
//   4 bits: 28672 x 4096 23.7 -> 15.9 (10.1), 6144 x 4096 8.9 -> 6.0 (2.2), 4096 x 4096 6.7 ->
//     4.9 (1.4), 4096 x 14336 17.4 -> 10.5 (5.0);
//   int8: 28672 x 4096 26.5 -> 22.0 (18.9), 6144 x 4096 9.6 -> 7.3 (4.1), 4096 x 14336 16.0 ->
//     12.2 (9.5), 2048 x 8192 8.6 -> 5.8 (2.7), 32000 x 2048 15.0 -> 13.7 (10.6);
//   bf16: 14336 x 4096 gated 41.7 -> 36.9 (37.9), 8192 x 2048 gated 15.7 -> 13.0 (10.8), 2048 x
//     8192 11.4 -> 7.7 (5.4), 2048 x 2048 5.1 -> 4.0 (1.4), 32000 x 2048 27.8 -> 22.5 (21.1).
// With the norm a product takes 0.3 to 0.7 us more, with rotation and cache write 0.5 to 1.3,
// where launches of their own took 2 to 4 each: a llama-1b step 412 -> 365 us, a llama-3-8b
// one in 4 bits, whose gate is in the product now, 604 -> 451.
// With two rows the same way is no faster (4 bits 28672 x 4096 23.7, bf16 4096 x 4096 9.9
// against 8.8).

#include "common.h"
#include "moe_tiles.h"

namespace {

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf2_t;

constexpr int kRows = 4;    // of W, a wave

DEVINLINE float dot2(unsigned a, unsigned b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2_t, a),
                                         __builtin_bit_cast(bf2_t, b), c, false);
}

// Ahead of the product: y = W rmsnorm(x + residual).  Every workgroup makes the row for itself
// (the sum rounded to bf16 as the norm's own launch leaves it, norm.hip; the first workgroup
// writes it) and multiplies W by sum * weight, rounded once as a normed row would be; what the
// squares say goes onto the f32 results, so that no thread waits for it before the product.
struct RowNorm {
  const __hip_bfloat16* residual;   // [K] or null
  __hip_bfloat16* sum;              // [K], not `residual`
  const __hip_bfloat16* weight;     // [K]; null: x as it is
  float eps;
};

// After the product of a step's query, key and value rows: queries turned, keys turned and
// values written into the cache (elementwise.hip).
struct RowTurn {
  const long* position;             // [1]
  const long* slot;                 // [1], negative: nothing is written
  const float* cos_sin;             // [positions, head size]
  unsigned char* k_cache;           // [slots, kv heads, head size]
  unsigned char* v_cache;
  int heads, kv_heads, shift;       // half a head: 1 << shift rows
  bool fp8;
};

enum RowMode { kRowPlain = 0, kRowGated = 1, kRowTurn = 2 };

// MODE: plain takes four neighbouring rows of W a wave, gated two of each half of W, turn two
// of each half of a head.  KS: waves that K is dealt to, the others take other rows of W.
template <int QB, int MODE, int KS, bool NORM, int kWaves>
__global__ __launch_bounds__(64 * kWaves, 4) void gemm_row_kernel(
    __hip_bfloat16* __restrict__ y,         // [N] (turn: the queries)
    const __hip_bfloat16* __restrict__ x,   // [K]
    const unsigned char* __restrict__ w,    // [(gated ? 2 : 1) * N, K]
    const float* __restrict__ scale,        // [rows of w] (8 bits) | [., K / 128] (4 bits)
    const int N, const int K, const RowNorm norm, const RowTurn turns) {
  constexpr int PER = 128 / QB;             // weights of a lane's 16 bytes
  constexpr int CPL = PER / 8;              // 16-byte chunks of x that go with them
  constexpr int SEG = 64 * PER;             // inputs of a wave's load
  constexpr bool PAIR = MODE != kRowPlain;
  constexpr int OUT = PAIR ? kRows / 2 : kRows, RS = kWaves / KS, COLS = RS * OUT;
  extern __shared__ __align__(16) char lds[];   // x [segments, CPL, 64] chunks
  __shared__ float sums[2][kWaves][kRows];
  __shared__ float squares[kWaves];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // addresses are scalars
  const int ks = wave % KS, rs = wave / KS;
  const int segs = (K + SEG - 1) / SEG;
  const int blocks = (MODE == kRowTurn ? N / 2 : N) / COLS;
  const long row_bytes = (long)K * QB / 8;
  const int far = MODE == kRowTurn ? 1 << turns.shift : N;   // rows between the halves
  // the first row of W of a block
  auto first_row = [&](int block) {
    const int at = block * COLS;
    return MODE == kRowTurn ? (at >> turns.shift << (turns.shift + 1)) + (at & (far - 1)) : at;
  };

  // (both waited for behind the row, which takes as long)
  long position = 0, slot = 0;
  if constexpr (MODE == kRowTurn) {
    position = *turns.position;
    slot = *turns.slot;
  }

  // what this thread stages first of x is asked for ahead of W, which takes longer
  const int chunks = segs * 64 * CPL;       // of x, past K zero
  constexpr int HELD = 2, STRIDE = 64 * kWaves;
  u32x4_t xv[HELD], rv[NORM ? HELD : 1], nv[NORM ? HELD : 1];
  auto fetch = [&](int c0, const __hip_bfloat16* from, u32x4_t* to) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const int c = c0 + i * STRIDE;
      to[i] = u32x4_t{};
      if (c * 8 < K) to[i] = *reinterpret_cast<const u32x4_t*>(from + c * 8);
    }
  };
  fetch(threadIdx.x, x, xv);
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) rv[i] = u32x4_t{};
    if (norm.residual != nullptr) fetch(threadIdx.x, norm.residual, rv);
    fetch(threadIdx.x, norm.weight, nv);
  }

  // a wave's loads, of segment `at_seg` of its rows of block `at`: with 4 bits, which take
  // longer to unpack, two are on their way (28672 x 4096 16.3 -> 15.8 us, 4096 x 4096 5.4 ->
  // 5.0; int8 22.5 -> 23.7, bf16 38.6 -> 39.7)
  struct Held {
    u32x4_t w[kRows];
    float s[QB == 4 ? kRows : 1];
  };
  constexpr bool DEEP = QB == 4;
  Held ta, tb;
  int at = blockIdx.x, at_seg = ks;
  auto load = [&](Held& t) {
    if (at >= blocks) return;
    const bool in = at_seg * SEG + lane * PER < K;   // K is a multiple of a lane's share
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const long n = first_row(at) + rs * OUT + (PAIR && r >= OUT ? far + r - OUT : r);
      const unsigned char* row = w + n * row_bytes + (long)at_seg * 1024;
      t.w[r] = u32x4_t{};
      if (in)
        t.w[r] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4_t*>(row + (unsigned)lane * 16));
      if constexpr (QB == 4) {
        const float* group = scale + n * (K / 128) + at_seg * (SEG / 128);
        t.s[r] = in ? group[(unsigned)lane / 4] : 0.f;
      }
    }
    at_seg += KS;
    if (at_seg >= segs) {
      at_seg = ks;
      at += gridDim.x;
    }
  };
  load(ta);
  if constexpr (DEEP) load(tb);

  u32x4_t* xs = reinterpret_cast<u32x4_t*>(lds);
  auto place = [&](int c) {
    const int in = c % (64 * CPL);
    return c - in + in % CPL * 64 + in / CPL;
  };
  auto stage = [&](int c, u32x4_t v) {
    if constexpr (QB == 4) {   // inputs 0 4 1 5 2 6 3 7, as the weights are unpacked
      const u32x4_t o = v;
      v[0] = __builtin_amdgcn_perm(o[2], o[0], 0x05040100);
      v[1] = __builtin_amdgcn_perm(o[2], o[0], 0x07060302);
      v[2] = __builtin_amdgcn_perm(o[3], o[1], 0x05040100);
      v[3] = __builtin_amdgcn_perm(o[3], o[1], 0x07060302);
    }
    xs[place(c)] = v;
  };
  union Chunk { u32x4_t u; __hip_bfloat16 h[8]; };
  float ss = 0.f;
  // what is left of a long row, more at a time (14336 inputs, 4 bits: 12.7 -> 11.9 us)
  if constexpr (!NORM) {
    constexpr int MORE = 5;
#pragma unroll 1
    for (int c0 = HELD * STRIDE + threadIdx.x; c0 < chunks; c0 += MORE * STRIDE) {
      u32x4_t v[MORE];
#pragma unroll
      for (int i = 0; i < MORE; ++i) {
        const int c = c0 + i * STRIDE;
        v[i] = u32x4_t{};
        if (c * 8 < K) v[i] = *reinterpret_cast<const u32x4_t*>(x + c * 8);
      }
#pragma unroll
      for (int i = 0; i < MORE; ++i)
        if (c0 + i * STRIDE < chunks) stage(c0 + i * STRIDE, v[i]);
    }
  }
#pragma unroll 1
  for (int c0 = threadIdx.x; c0 < (NORM ? chunks : HELD * STRIDE); c0 += HELD * STRIDE) {
    if (c0 != threadIdx.x) {
      fetch(c0, x, xv);
      if constexpr (NORM) {
        if (norm.residual != nullptr) fetch(c0, norm.residual, rv);
        fetch(c0, norm.weight, nv);
      }
    }
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const int c = c0 + i * STRIDE;
      if (c >= chunks) continue;
      if constexpr (NORM) {
        Chunk v, r, g;
        v.u = xv[i];
        r.u = rv[i];
        g.u = nv[i];
        if (norm.residual != nullptr) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            v.h[j] = __float2bfloat16(__bfloat162float(v.h[j]) + __bfloat162float(r.h[j]));
          if (blockIdx.x == 0 && c * 8 < K) *reinterpret_cast<u32x4_t*>(norm.sum + c * 8) = v.u;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float f = __bfloat162float(v.h[j]);
          ss += f * f;
          v.h[j] = __float2bfloat16(f * __bfloat162float(g.h[j]));
        }
        xv[i] = v.u;
      }
      stage(c, xv[i]);
    }
  }
  if constexpr (NORM) {
    ss = wave_reduce_sum(ss);
    if (lane == 0) squares[wave] = ss;
  }
  // what a block's results need is on its way beside its weights
  float cosine = 1.f, sine = 0.f;
  auto angles = [&](int block) {
    const int p = block * COLS + threadIdx.x;
    if (threadIdx.x < COLS && p >> turns.shift < turns.heads + turns.kv_heads) {
      const float* cs = turns.cos_sin + position * 2 * far + (p & (far - 1));
      cosine = cs[0];
      sine = cs[far];
    }
  };
  if constexpr (MODE == kRowTurn) angles(blockIdx.x);
  __syncthreads();
  float inv = 1.f;
  if constexpr (NORM) {
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) ss += squares[i];
    inv = rsqrtf(ss / K + norm.eps);
  }

  // (in a register: and-or takes one constant from elsewhere)
  unsigned eights = 0x41004100u;
  if constexpr (QB == 4) asm volatile("" : "+v"(eights));

  int turn = 0, block = blockIdx.x, seg = ks;
  float acc[kRows] = {}, row_scale = QB == 4 ? 2.f : 1.f, far_scale = row_scale;
  auto step = [&](Held& t) {
    if (seg == ks) {   // a new block
      if constexpr (MODE == kRowTurn)
        if (block != blockIdx.x) angles(block);
      if constexpr (QB == 8) {
        if (threadIdx.x < COLS) {
          row_scale = scale[first_row(block) + threadIdx.x];
          if constexpr (PAIR) far_scale = scale[first_row(block) + threadIdx.x + far];
        }
      }
#pragma unroll
      for (int r = 0; r < kRows; ++r) acc[r] = 0.f;
    }
    if (seg < segs) {
      u32x4_t q[kRows];
      float s[QB == 4 ? kRows : 1];
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        q[r] = t.w[r];
        if constexpr (QB == 4) s[r] = t.s[r];
        // whole registers: the compiler would carry every weight of the next load by itself
        if constexpr (QB != 16)
#pragma unroll
          for (int d = 0; d < 4; ++d) asm volatile("" : "+v"(q[r][d]));
      }
      load(t);
      float part[kRows] = {}, base = 0.f;
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        const u32x4_t xc = xs[(seg * CPL + j) * 64 + lane];
        if constexpr (QB == 4) {
#pragma unroll
          for (int d = 0; d < 4; ++d) base = dot2(xc[d], 0xc140c140u, base);   // -12
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            unsigned two;
            if constexpr (QB == 16) {
              two = q[r][d];
            } else if constexpr (QB == 8) {
              // whole numbers of 8 bits: the upper half of the float is all of it
              const unsigned four = q[r][2 * j + d / 2] >> (d % 2 * 16);
              const float a = (float)(signed char)(four & 0xff);
              const float b = (float)(signed char)((four >> 8) & 0xff);
              two = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
            } else {   // 8 + n / 2
              two =
                  ((d == 0 ? q[r][j] << 3 : q[r][j] >> (4 * d - 3)) & 0x00780078u) | eights;
            }
            float& to = QB == 4 ? part[r] : acc[r];
            to = dot2(xc[d], two, to);
          }
        // a chunk at a time: unpacked all at once the weights take twice the registers
        if constexpr (QB != 16) __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (QB == 4) {
#pragma unroll
        for (int r = 0; r < kRows; ++r) acc[r] = __builtin_fmaf(s[r], part[r] + base, acc[r]);
      }
    }
    seg += KS;
    if (seg < segs) return;

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
      float g = 0.f, u = 0.f;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        g += sums[turn][first + k][o];
        if constexpr (PAIR) u += sums[turn][first + k][OUT + o];
      }
      if constexpr (QB != 16 || NORM) {
        g *= row_scale * inv;
        u *= far_scale * inv;
      }
      const int n = block * COLS + threadIdx.x;
      if constexpr (MODE != kRowTurn) {
        y[n] = __float2bfloat16(moe::finish<MODE == kRowGated ? moe::kSilu : moe::kPlain>(g, u, 0.f));
      } else {
        const int head = n >> turns.shift, i = n & (far - 1), key = head - turns.heads;
        __hip_bfloat16 lo = __float2bfloat16(g), hi = __float2bfloat16(u);
        if (key < turns.kv_heads) {
          const float x1 = __bfloat162float(lo), x2 = __bfloat162float(hi);
          lo = __float2bfloat16(x1 * cosine - x2 * sine);
          hi = __float2bfloat16(x2 * cosine + x1 * sine);
        }
        if (key < 0) {
          y[head * 2 * far + i] = lo;
          y[head * 2 * far + far + i] = hi;
        } else if (slot >= 0) {
          const bool value = key >= turns.kv_heads;
          unsigned char* cache = value ? turns.v_cache : turns.k_cache;
          const long to =
              (slot * turns.kv_heads + key - (value ? turns.kv_heads : 0)) * 2 * far + i;
          if (turns.fp8) {
            const int two = __builtin_amdgcn_cvt_pk_fp8_f32(__bfloat162float(lo),
                                                            __bfloat162float(hi), 0, false);
            cache[to] = (unsigned char)two;
            cache[to + far] = (unsigned char)(two >> 8);
          } else {
            reinterpret_cast<__hip_bfloat16*>(cache)[to] = lo;
            reinterpret_cast<__hip_bfloat16*>(cache)[to + far] = hi;
          }
        }
      }
    }
    seg = ks;
    block += gridDim.x;
    turn ^= 1;
  };
  while (block < blocks) {
    step(ta);
    if constexpr (DEEP)
      if (block < blocks) step(tb);
  }
}

struct RowCall {
  __hip_bfloat16* y;
  const __hip_bfloat16* x;
  const void* w;
  const float* scale;
  int N, K;
  RowNorm norm;
  RowTurn turns;
  hipStream_t stream;
};

template <int QB, int MODE, int KS, bool NORM, int kWaves>
void launch(const RowCall& c) {
  constexpr int SEG = 64 * 128 / QB, COLS = kWaves / KS * (MODE == kRowPlain ? kRows : kRows / 2);
  static_assert(128 % COLS == 0 && 16 % COLS == 0, "whole workgroups, inside half a head");
  // sixteen waves a CU walk the rows (28672 x 4096 4 bits: 17.0 us, eight 19.1, all 19.2)
  constexpr int MOST = 256 * 16 / kWaves;
  const int blocks = (MODE == kRowTurn ? c.N / 2 : c.N) / COLS;
  hipLaunchKernelGGL((gemm_row_kernel<QB, MODE, KS, NORM, kWaves>),
                     dim3(blocks < MOST ? blocks : MOST), dim3(64 * kWaves), (c.K + SEG - 1) / SEG * SEG * 2, c.stream, c.y, c.x,
                     static_cast<const unsigned char*>(c.w), c.scale, c.N, c.K, c.norm, c.turns);
}

// The rows of W that the busiest CU has when workgroups take `cols` of N at a time.
int busiest(int N, int cols) { return (N / cols + 255) / 256 * cols; }

// How many workgroups share a CU's LDS, for the row that each keeps there, and whether that is fewer than
// four of four waves.
int resident(int K) { return 80 * 1024 / (K + 64); }
bool crowded(int K) { return resident(K) < 4; }

}  // namespace

// Waves of a workgroup, and over how many of them K is dealt: waves << 4 | those.  A function of sizes.
// With eight waves half as many workgroups stage x, and of long K more is asked for at once; K dealt to
// more waves leaves shorter chains where rows are few, to fewer less to add up and more rows that share
// x.  Workgroups that take more rows (16 by 8/2 and 4/1, 8 by 8/4 and 4/2, 4 by 4/4 and 8/8) leave CUs
// with fewer rows than others: `busiest`.  us, N x K, W/KS:
//   bf16, plain: up to 2048 rows all workgroups of 8/8 are there at once, 4/4 | 8/8: 2048 x 8192 8.70 | 7.78,
//     768 x 8192 6.01 | 4.97, 128 x 7168 5.46 | 4.17 (to 4096 inputs 8/8 loses 6 %); up to 4096 only
//     those of 4/4 are: 2176 x 10240 10.54 | 11.09, 2560 x 14336 14.5 | 14.8, 3072 x 8192 11.1 | 10.9, but
//     crowded, 2560 x 28672 33.8 | 26.1; past that neither are: 5120 x 8192 16.6 | 16.0, 4608 x 14336 24.7 |
//     23.0, 9216 x 14336 41.6 | 40.1, 7168 x 9216 22.2 | 22.7.  Many sums of eight waves are seen while K
//     is short, 4/4 | 8/8 | 8/4: 16384 x 8192 42.8 | 44.3 | 42.7, 8192 x 8192 23.3 | 23.4 | 23.1, 20480 x
//     7168 45.7 | .. | 44.5, 6144 x 8192 18.5 | 18.3 | 18.3, 16384 x 9216 47.2 | 46.8 | 45.7.
//     Gated, 4/4 | 4/2, two loads of K: 3072 x 1024 5.77 | 5.18; four: 8192 x 2048 13.5 | 12.4, 2048 x 2048
//     6.05 | 5.88, but 1024 x 2048 4.73 | 5.16; three, of which one of two waves has two: 8192 x 1280
//     10.3 | 9.6, 5120 x 1280 7.40 | 7.72, 2048 x 1280 5.14 | 5.37.  Long K, 4/4 | 8/4: 28672 x 8192 147.0 | 145.2,
//     2048 x 8192 15.2 | 13.4, 128 x 8192 7.00 | 6.78 (14336 x 4096 38.8 | 38.6).
//     Turned, 4/4 | 8/8 | 8/4: 1280 x 8192 8.52 | 7.69 | 8.24, 5120 x 8192 17.9 | 17.2 | 18.5, 6144 x 10240 23.8 |
//     22.6 | 22.4, 10240 x 8192 31.6 | 31.2 | 30.8 (6144 x 4096 10.8 | 11.2 | 11.2).
//   int8, plain, 4/4 | 8/4: 4096 x 14336 12.5 | 12.1, 2048 x 8192 6.2 | 5.8, 1280 x 14336 7.7 | 7.1, 10240 x
//     14336 25.7 | 24.6 (4096 x 4096 5.79 | 5.83); a CU with more rows: 256 x 14336 5.80 | 6.42, 2560 x
//     14336 9.6 | 10.2, 4608 x 8192 8.55 | 8.89; crowded, 3328 x 20480 17.6 | 13.4, 2560 x 28672
//     19.9 | 17.0.
//     Gated, a load of K, 4/2 | 4/1: 14336 x 1024 9.7 | 8.4, 512 x 1024 3.72 | 3.66; two: 8192 x 2048 9.0 |
//     8.5, 4096 x 2048 6.6 | 6.1, 5120 x 1280 6.0 | 6.6, 1024 x 2048 4.1 | 4.5.  Longer, 4/4 | 4/2: 14336 x 4096
//     22.2 | 20.8, 2048 x 4096 7.0 | 6.5, 512 x 4096 4.3 | 4.8, 1152 x 2560 5.2 | 5.4; 4/4 | 8/4: 28672 x
//     8192 73.4 | 72.0, 2048 x 8192 10.5 | 8.7, 128 x 8192 5.5 | 5.4.  Turned, 4/4 | 8/4: 6144 x 4096 8.0 |
//     7.4, 10240 x 8192 17.4 | 16.2, 3072 x 4096 6.36 | 6.52.
//   4 bits (a load covers 2048 inputs), plain, K past three loads.  Up to 2047 rows, 4/4 | 8/8: 1024 x 8192
//     4.30 | 4.02, 128 x 28672 7.3 | 6.5.  Four loads, 4/4 | 8/4, all workgroups there at once: 4096 x 8192
//     7.31 | 6.75, 2048 x 8192 5.44 | 5.02; more rows, 4/4 | 4/2 | 8/2: 5120 x 8192 8.4 | 8.8 | 9.7, 6144 x
//     7168 9.0 | 8.8 | 9.3, 8192 x 8192 11.1 | 10.5 | 10.8, 10240 x 8192 12.9 | 12.1 | 13.6, 28672 x 8192
//     27.0 by 4/1 | 25.4 | 27.6.  Longer, 8/2 where CUs have as many rows as with fewer a workgroup, 4/4 | 4/2 | 8/2:
//     4096 x 14336 10.4 | 10.0 | 10.2, 7680 x 14336 16.1 | .. | 14.6, 8192 x 14336 16.2 | 15.6 | 14.9, but
//     4608 x 14336 11.5 | 12.2 | 13.5, 5120 x 10240 9.6 | 10.2 | 10.7, 10240 x 14336 18.0 | 17.6 | 18.6, 14336 x 14336 22.9 | 22.9 |
//     24.5, 2560 x 14336 8.8 by 4/4 | 9.1; past 16384, 4/1 | 8/2: 57344 x 14336 71 | 75, 28672 x 14336 39.1 | 39.2.
//     Crowded, 4/4 | 8/2 | 8/4 | 8/8: 8192 x 28672 31 | 24.6 | 26.6 | 27.3, 4096 x 28672 19.7 | 14.9 | 16.3 | 16.8,
//     6144 x 28672 25.1 | 23.0 | 20.7 | 22.3, 5120 x 28672 22.8 | 22.8 | 20.1 | 19.0.
//     Shorter K, and with pairs: rows go first where they are many (14336 x 4096 gated 4/1 16.9, 4/2 17.9;
//     2048 x 8192 4/1 7.0, 4/2 5.5).
int gemm_row_form(int qbits, int mode, int N, int K) {
  constexpr int k41 = 0x41, k42 = 0x42, k44 = 0x44, k82 = 0x82, k84 = 0x84, k88 = 0x88;
  const int r4 = busiest(N, 4), r8 = busiest(N, 8), r16 = busiest(N, 16);
  if (qbits == 16) {
    if (mode == kRowGated)
      return K >= 8192 ? k84
             : K <= 1024 || (K <= 2048 && N >= (K > 1536 ? 2048 : 8192)) ? k42 : k44;
    if (mode == kRowTurn) return K < 8192 ? k44 : N <= 5120 ? k88 : k84;
    if (K < 7168 || (N > 2048 && N < 4096 && !crowded(K))) return k44;
    return N >= 8192 && K <= 8192 ? k84 : k88;
  }
  if (qbits == 8) {
    if (mode == kRowGated) {
      if (K <= 2048) return K <= 1024 || N >= (K > 1792 ? 3584 : 8192) ? k41 : k42;
      return K >= 8192 ? k84 : N >= 1280 ? k42 : k44;
    }
    if (K <= 2048) return k42;
    if (mode == kRowTurn) return K >= 4096 && N >= 6144 ? k84 : k44;
    return K >= 7168 && (r8 <= r4 || (crowded(K) && r4 > 4 * resident(K))) ? k84 : k44;
  }
  const int rows = mode == kRowGated ? 2 * N : N;
  if (mode != kRowPlain || K <= 2048 * 3)
    return mode != kRowPlain && K > 2048 * 3 && rows <= 8192 ? k44
           : K > 2048 && rows <= 16384                       ? k42 : k41;
  if (N < 2048) return k88;
  if (K <= 8192) return N <= 4096 ? k84 : N > 8192 || r8 <= r4 ? k42 : k44;
  if (crowded(K)) return r16 <= r8 ? k82 : r8 <= r4 ? k84 : k88;
  if (N > 16384) return k41;
  if (r16 <= r8 && (N > 4096 || r16 <= r4)) return k82;
  if (N <= 4096) return r8 <= r4 ? k84 : k44;
  return N > 8192 || r8 <= r4 ? k42 : k44;
}

namespace {

template <int MODE, bool NORM>
void launch_bits(const RowCall& c, int qbits) {
  const int form = gemm_row_form(qbits, MODE, c.N, c.K);
#define GO(QB, W, KS) if (qbits == QB && form == (W << 4 | KS)) return launch<QB, MODE, KS, NORM, W>(c)
  GO(16, 4, 4);
  GO(16, 8, 4);
  GO(8, 4, 4);
  GO(8, 4, 2);
  GO(8, 8, 4);
  GO(4, 4, 4);
  GO(4, 4, 2);
  if constexpr (MODE == kRowGated) {
    GO(16, 4, 2);
    GO(8, 4, 1);
  } else {
    GO(16, 8, 8);
  }
  if constexpr (MODE == kRowPlain) {
    GO(4, 8, 2);
    GO(4, 8, 4);
    GO(4, 8, 8);
  }
  launch<4, MODE, 1, NORM, 4>(c);
#undef GO
}

}  // namespace

// x is kept in LDS
bool gemm_row_fits(int K) { return K <= 28672; }

// N % 128 == 0, K % 64 == 0 (rounded weights: K % 128 == 0)
void launch_gemm_row(__hip_bfloat16* y, const __hip_bfloat16* x, const void* w,
                     const float* scale, int qbits, int N, int K, bool gated,
                     hipStream_t stream) {
  const RowCall c{y, x, w, scale, N, K, RowNorm{}, RowTurn{}, stream};
  if (gated) launch_bits<kRowGated, false>(c, qbits);
  else launch_bits<kRowPlain, false>(c, qbits);
}

// y = silu(n Wg^T) * (n Wu^T), n = rmsnorm(x + residual) * weight, sum = x + residual (without
// a residual: of x, and no sum).
void launch_gemm_row_norm_gated(__hip_bfloat16* y, __hip_bfloat16* sum, const __hip_bfloat16* x,
                                const __hip_bfloat16* residual, const __hip_bfloat16* weight,
                                float eps, const void* w, const float* scale, int qbits, int N,
                                int K, hipStream_t stream) {
  launch_bits<kRowGated, true>(
      RowCall{y, x, w, scale, N, K, RowNorm{residual, sum, weight, eps}, RowTurn{}, stream}, qbits);
}

// The same norm, then the rows of W for queries, keys and values of heads of 2 << shift
// (shift >= 4): q = the queries turned; keys turned and values go into the cache.
void launch_gemm_row_norm_turn(__hip_bfloat16* q, __hip_bfloat16* sum, const __hip_bfloat16* x,
                               const __hip_bfloat16* residual, const __hip_bfloat16* weight,
                               float eps, const void* w, const float* scale, int qbits, int K,
                               const long* position, const long* slot, const float* cos_sin,
                               void* k_cache, void* v_cache, int heads, int kv_heads, int shift,
                               bool fp8, hipStream_t stream) {
  const RowTurn turns{position, slot, cos_sin, static_cast<unsigned char*>(k_cache),
                      static_cast<unsigned char*>(v_cache), heads, kv_heads, shift, fp8};
  launch_bits<kRowTurn, true>(RowCall{q, x, w, scale, (heads + 2 * kv_heads) << (shift + 1), K,
                                      RowNorm{residual, sum, weight, eps}, turns, stream},
                              qbits);
}
