// Paged causal prompt attention: bf16 or e4m3 cache, heads of 64 or 128.
//
// A workgroup takes NW waves of 32 query rows of one key head: as many of its query heads
// as divide the waves, and the tokens that are left over of them, so that the keys of a
// tile serve all heads and the rows of a workgroup end at nearly the same key.  Tiles of
// 64 keys and values are staged once for all of them, bf16 straight HBM -> LDS
// (global_load_lds), the block ids a tile ahead of the loads.
//
// v_mfma_f32_32x32x16_bf16 takes S^T = K Q^T, so a lane keeps one query's statistics and
// accumulators; 16 keys of the scores enter the second product in the order the score
// layout has them, so probabilities are packed where they are, and the values come back
// transposed (ds_read_b64_tr_b16).
//
// Bound by what a SIMD issues: a tile of 64 keys (heads of 128) takes a wave 32 products of 32
// clocks, of which each keeps the vector unit for about 12, and some 1050 clocks of exponentials
// (16 each), sums and packing.  With eight waves the two of a SIMD take turns, one making
// probabilities while the other multiplies: 2 x 1550 clocks of 2 x 1050 + 64 x 12.  What that took:
//  - block ids and addresses on the scalar unit.  By the lanes they were 500 clocks a tile,
//    and ids that went through vector memory had the compiler wait for the whole next tile.
//  - three tiles of keys and of values in LDS, so that a turn's first fragments are read ahead of
//    its barrier; addresses are constants then, no vector instruction lies between the products.
//  - reads in batches: with transposed ones among them the compiler waits for all.
//  - chunks of values turned so that sixteen lanes of a transposed read lie in different banks
//    (2.7 -> 1.9 clocks a read of a full LDS).
// Fewer waves, where a workgroup's are alone or two workgroups share a CU, and eight that find their
// rows by the lanes, but in bf16 heads of 128: products of the next tile's scores between this
// one's exponentials.
//
// Measured (MI355X, 32/8 heads of 128, keys and queries of variance 1, before -> after): 3500
// tokens of 7 prompts after 700 each, bf16: 86 -> 74 us; one prompt of 8192 tokens 580 -> 522 us (1050
// TFLOP/s; e4m3 605 -> 555), 3000 tokens 114 -> 100, 512 tokens after 5000 75 -> 67.  Turns alone, with
// the lanes' addresses, were worth 1 %.  Blocks that a wave's load does not fit (under 4 to 16 rows, or
// no power of two) leave the addresses to the lanes: blocks of 24, 3000 tokens 120 -> 111, e4m3 121 ->
// 120, 33 tokens 7.0 -> 7.1.
// On the way here: eight waves of one head (256 tokens) leave early rows' waves idle; register
// staging 630 us of 564; transposed reads as asm 584; results stored in 8 bytes a lane instead of
// 16: 24 tokens 7.0 us instead of 6.2.

#include "common.h"
#include <float.h>
#include <algorithm>
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

namespace {

constexpr int kTile = 64;   // keys of a step
// A part is no shorter: few tokens after a long context are a chain of tiles, and what a part leaves is
// little (8 prompts of 2 tokens after 600 in 1 | 3 parts: 18.4 | 13.3 us, e4m3 21.3 | 14.6; 64 after 2000
// in 5 | 8: 22.0 | 20.7, e4m3 23.7 | 22.0)
constexpr int kMinTiles = 3;
constexpr float kLog2e = 1.4426950408889634f;
// A maximum that grew by less than this (log2) is not followed: sums and probabilities
// stay in range, their relative precision is the same.
constexpr float kDefer = 11.5f;

typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf2_t;
DEVINLINE unsigned pack_bf16(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2_t{a, b}, bf2_t));
}

typedef __attribute__((address_space(3))) bf16x8_t lds_bf16x8_t;

// Through a restrict parameter: without it the compiler takes the builtin for a read of
// whatever is on its way to LDS, and has it wait for the loads of the next tile.
DEVINLINE s16x4_t read_transposed(lds_s16x4_t* __restrict__ at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(at);
}

// 16-byte chunk c of row r of a tile lies at chunk c ^ swizzle(r).  Keys: the 16 rows of
// equal chunks cover all banks.  Values: pairs of chunks stay pairs, the four rows of a
// transposed read lie in different banks; PAIRS: two by two only, which is as good where rows found by
// the lanes are widened on their way to LDS (4 prompts of 500 after 700, e4m3, blocks of 24: 76.1 | 73.0).
template <int HD> DEVINLINE int k_swizzle(int r) { return HD == 128 ? r & 15 : (r >> 1) & 7; }
template <int HD, bool PAIRS> DEVINLINE int v_swizzle(int r) {
  if (PAIRS) return HD == 128 ? (r & 7) * 2 : ((r >> 1) & 3) * 2;
  return HD == 128 ? (r & 3) * 4 : (r & 2) * 2;
}

// tiles of keys that one part takes
DEVINLINE int tiles_per_part(int tiles, int parts) {
  return max(kMinTiles, (tiles + parts - 1) / parts);
}

// Whether the two waves of a SIMD take turns: not where the lanes find their rows and little is won by
// it (us, two tiles in LDS | in turns, blocks of 24: e4m3, 512 tokens after 5000 80 | 82, 4 prompts of
// 500 after 700 76 | 79; heads of 64 21.4 | 22.6; bf16 heads of 128 76 | 72)
template <int HD, typename CT, int NW, bool EVEN>
constexpr bool kTurns = NW == 8 && (EVEN || (sizeof(CT) == 2 && HD == 128));

// The LDS of a workgroup, an array of BYTES or, FROM_0, of the launch's size, which has the address 0: a
// static array's is not known to be that, and is added to the lanes' (rows found by the lanes, us, static |
// from 0: 33 tokens e4m3 8.2 | 7.8, 100 after 200 17.2 | 16.2, bf16 14.1 | 13.8; but in turns, where no
// addresses are left, e4m3, 512 after 5000 70 | 71, 4 prompts of 500 after 700 66 | 67).
template <int BYTES, bool FROM_0> DEVINLINE char* shared_bytes() {
  if constexpr (FROM_0) {
    extern __shared__ __align__(16) char given[];
    return given;
  } else {
    __shared__ __align__(16) char own[BYTES];
    return own;
  }
}

// EVEN: cache blocks are a multiple of the rows of a wave's load (and a power of two), so that
// these have one block
template <int HD, typename CT, int NW, bool EVEN>
__global__ __launch_bounds__(NW * 64, 2) void paged_prefill_tile_kernel(
    __hip_bfloat16* __restrict__ out,         // [total_q, nheads, HD]
    const __hip_bfloat16* __restrict__ q,     // [total_q, nheads, HD]
    const CT* __restrict__ k_cache,           // [blocks, block_size, kvh, HD]
    const CT* __restrict__ v_cache,
    const int* __restrict__ block_tables,     // [nseq, max_blocks]
    const int* __restrict__ query_start_loc,  // [nseq + 1]
    const int* __restrict__ seq_lens,         // [nseq]
    const float scale_log2, const int nheads, const int kvh, const int heads,  // of a workgroup
    const int block_size, const int block_shift, const int max_blocks, const int parts,
    float* __restrict__ part_acc,             // [parts, total_q, nheads, HD] (parts > 1)
    float* __restrict__ part_ml) {            // [parts, total_q, nheads, 2]  (parts > 1)
  constexpr bool FP8 = sizeof(CT) == 1;
  constexpr int KS = HD / 16;          // contraction steps of a score tile
  constexpr int DT = HD / 32;          // 32-wide tiles of the result
  constexpr int CPR = HD / 8;          // 16-byte chunks of a row in LDS
  constexpr int LPR = HD * sizeof(CT) / 16;   // lanes a cache row takes
  constexpr int RPP = 64 / LPR;               // rows of a wave's load
  constexpr int PASS = kTile / RPP / NW;      // loads of a thread, keys or values
  constexpr int BYTES = kTile * HD * 2;
  static_assert(PASS * RPP * NW == kTile, "whole passes");
  constexpr bool TURNS = kTurns<HD, CT, NW, EVEN>;

  const int seq = blockIdx.y;
  const int q_start = query_start_loc[seq];
  const int q_len = query_start_loc[seq + 1] - q_start;
  const int seq_len = seq_lens[seq];
  const int tokens = NW / heads * 32;
  // the last tokens see the most keys: they go first
  const int tile = (q_len + tokens - 1) / tokens - 1 - (int)blockIdx.z / parts;
  if (tile < 0) return;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int scalar_wave = __builtin_amdgcn_readfirstlane(wave);
  const int col = lane & 31, half = lane >> 5;
  const int group = nheads / kvh, per_kv = group / heads;   // workgroups of a key head
  const int kv_head = blockIdx.x / per_kv;
  const int head = kv_head * group + blockIdx.x % per_kv * heads + wave % heads;
  const int token0 = tile * tokens + wave / heads * 32;
  const int token = min(token0 + col, q_len - 1);
  const int past = seq_len - q_len;
  const int keys = min(seq_len, past + min((tile + 1) * tokens, q_len));
  const int tiles = (keys + kTile - 1) / kTile, per = tiles_per_part(tiles, parts);
  const int first = blockIdx.z % parts * per;
  // no keys at all: part 0 writes the zeros
  if (first >= tiles && first > 0) return;
  const int n = min(per, tiles - first), origin = first * kTile;
  // positions from the part's first key on
  const int q_pos = past + token - origin;
  const int wave_min = past + token0 - origin;
  const int wave_max = token0 < q_len ? past + min(token0 + 31, q_len - 1) - origin : -1;

  constexpr int BUFS = TURNS ? 3 : 2;
  char* const lds_all = shared_bytes<2 * BUFS * BYTES, !TURNS>();   // tiles of keys, then of values
  char* const k_lds[2] = {lds_all, lds_all + BYTES};
  char* const v_lds[2] = {lds_all + BUFS * BYTES, lds_all + (BUFS + 1) * BYTES};

  const __hip_bfloat16* q_row = q + ((long)(q_start + token) * nheads + head) * HD + half * 8;
  bf16x8_t qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const bf16x8_t*>(q_row + ks * 16);

  // ---- staging -----------------------------------------------------------
  const int* table = block_tables + (long)seq * max_blocks;
  const long row_bytes = (long)kvh * HD * sizeof(CT);
  const char* k_at = reinterpret_cast<const char*>(k_cache) + kv_head * HD * sizeof(CT);
  const char* v_at = reinterpret_cast<const char*>(v_cache) + kv_head * HD * sizeof(CT);
  auto row_of = [&](int ps) { return (ps * NW + wave) * RPP + lane / LPR; };
  // Block ids of a tile's keys (past the end: of the last key), and what they lead to: apart, so
  // that nothing waits for the ids before the next step.  With EVEN blocks both are the wave's, on
  // the scalar unit: a lane by itself takes 500 of the vector unit's clocks a tile for them,
  // half as much as for its probabilities.
  struct Place {       // of a wave's load in the cache
    std::conditional_t<EVEN, long, int> at;   // where its first row begins; else: the lane's row
    int last;   // EVEN: rows past it are this one again
  };
  auto pos_of = [&](int ps, int t) {
    return min(origin + t * kTile + (EVEN ? (ps * NW + scalar_wave) * RPP : row_of(ps)), keys - 1);
  };
  auto page_of = [&](int pos) {
    return EVEN || block_shift >= 0 ? pos >> block_shift : pos / block_size;
  };
  auto ids_of = [&](int (&ids)[PASS], int t) {
#pragma unroll
    for (int ps = 0; ps < PASS; ++ps) ids[ps] = table[page_of(pos_of(ps, t))];
  };
  // (ahead of a tile's loads: behind them the compiler has all of these land before it touches
  // the ids, a memory latency in every tile)
  auto places_of = [&](Place (&places)[PASS], const int (&ids)[PASS], int t) {
#pragma unroll
    for (int ps = 0; ps < PASS; ++ps) {
      const int pos = pos_of(ps, t), in = pos - page_of(pos) * block_size;
      if constexpr (EVEN) {
        places[ps] = Place{(((long)ids[ps] << block_shift) + in) * row_bytes, keys - 1 - pos};
      } else {
        int row = ids[ps] * block_size + in;
        if constexpr (TURNS) asm volatile("" : "+v"(row));
        places[ps] = Place{row, 0};
      }
    }
  };
  u32x4_t kr[FP8 ? PASS : 1], vr[FP8 ? PASS : 1];
  auto issue = [&](const char* cache, const Place (&places)[PASS], char* lds, auto& regs,
                   auto swizzle) {
#pragma unroll
    for (int ps = 0; ps < PASS; ++ps) {
      const char* row;
      unsigned in = (FP8 ? lane % LPR : (lane % LPR) ^ swizzle(row_of(ps))) * 16;
      if constexpr (EVEN) {
        row = cache + places[ps].at;
        in += __umul24(min(lane / LPR, places[ps].last), (unsigned)row_bytes);
      } else {
        row = cache + places[ps].at * row_bytes;
      }
      if constexpr (FP8)
        regs[ps] = *reinterpret_cast<const u32x4_t*>(row + in);
      else
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) unsigned*)(row + in),
            (__attribute__((address_space(3))) unsigned*)(lds + (ps * NW + scalar_wave) * 1024), 16,
            0, 0);
    }
  };
  auto unpack = [&](char* lds, const auto& regs, auto swizzle) {
#pragma unroll
    for (int ps = 0; ps < PASS; ++ps)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x2_vec_t u;
        u[0] = regs[ps][2 * h];
        u[1] = regs[ps][2 * h + 1];
        const int r = row_of(ps);
        *reinterpret_cast<bf16x8_vec_t*>(
            lds + r * HD * 2 + ((lane % LPR * 2 + h) ^ swizzle(r)) * 16) = fp8x8_to_bf16x8(u);
      }
  };
  auto k_swz = [](int r) { return k_swizzle<HD>(r); };
  auto v_swz = [](int r) { return v_swizzle<HD, FP8 && !EVEN>(r); };
  auto block_meet = [&] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // own loads have landed (or are written to LDS), everybody's have
  auto meet = [&] {
    if constexpr (FP8) {
      __syncthreads();
    } else {
      __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
      block_meet();
    }
  };

  // ---- the two products ----------------------------------------------------
  float m_state = -FLT_MAX, l_state = 0.f;   // of query `col`, raw scores; l: this half's keys
  f32x16_t acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16_t{};

  // LDS addresses in the first tile of keys and of values; kept out of the compiler's sight,
  // which would rather compute them again than keep them (where there are registers for it)
  constexpr bool KEEP = !FP8 && NW == 8;
  unsigned k_lane[KS], v_lane[DT], lds_at = 0;
  if constexpr (TURNS)
    lds_at = (unsigned)(__SIZE_TYPE__)(__attribute__((address_space(3))) char*)lds_all;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    k_lane[ks] = lds_at + col * HD * 2 + ((ks * 2 + half) ^ k_swizzle<HD>(col)) * 16;
    if constexpr (KEEP) asm volatile("" : "+v"(k_lane[ks]));
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int i = lane & 15, side = lane >> 4 & 1, r = half * 4 + (i >> 2);
    v_lane[dt] = lds_at + BUFS * BYTES + r * HD * 2 +
                 (((dt * 2 + side) * 2 + ((i & 3) >> 1)) ^ v_swizzle<HD, FP8 && !EVEN>(r)) * 16 + (i & 1) * 8;
    if constexpr (KEEP) asm volatile("" : "+v"(v_lane[dt]));
  }
  auto key_frag = [&](int at, int g) {   // g: 32-key half g % 2, 16 dims g / 2
    return *(const lds_bf16x8_t*)(k_lane[g >> 1] + (at + (g & 1) * 32 * HD * 2));
  };
  // next = scores of the tile in lds; between its products, work(i), i = 0..15
  auto scores = [&](f32x16_t (&next)[2], int at, auto work) {
    constexpr int AHEAD = 3;
    bf16x8_t kf[AHEAD];
#pragma unroll
    for (int g = 0; g < AHEAD; ++g) kf[g] = key_frag(at, g);
#pragma unroll
    for (int g = 0; g < 2 * KS; ++g) {
      next[g & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          kf[g % AHEAD], qf[g >> 1], g < 2 ? f32x16_t{} : next[g & 1], 0, 0, 0);
      if (g + AHEAD < 2 * KS) kf[g % AHEAD] = key_frag(at, g + AHEAD);
#pragma unroll
      for (int i = 0; i < 8 / KS; ++i) work(g * (8 / KS) + i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const float defer = kDefer / scale_log2;
  // lane: keys base + 32 kb + 8 (r / 4) + 4 half + r % 4 of query col
  auto follow = [&](f32x16_t (&s)[2], const int base) {
    if (base + kTile - 1 > wave_min) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (base + kb * 32 + (r >> 2) * 8 + half * 4 + (r & 3) > q_pos) s[kb][r] = -FLT_MAX;
    }
    float big = fmaxf(s[0][0], s[1][0]);
#pragma unroll
    for (int r = 1; r < 16; ++r) big = fmaxf(fmaxf(big, s[0][r]), s[1][r]);
    const auto sides = __builtin_amdgcn_permlane32_swap(
        __builtin_bit_cast(unsigned, big), __builtin_bit_cast(unsigned, big), false, false);
    big = fmaxf(__builtin_bit_cast(float, sides[0]), __builtin_bit_cast(float, sides[1]));
    if (!__all(m_state != -FLT_MAX && big <= m_state + defer)) {
      const float m_new = fmaxf(m_state, big);
      const float f = __builtin_amdgcn_exp2f((m_state - m_new) * scale_log2);
      l_state *= f;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] *= f;
      m_state = m_new;
    }
  };
  union Probs { unsigned u[4]; bf16x8_t v; };
  // two of 32 probabilities
  float bias;
  auto weigh = [&](const f32x16_t (&s)[2], Probs (&p)[4], int i) {
    const int kb = i >> 3, r = i % 8 * 2;
    const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], scale_log2, bias));
    const float b = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r + 1], scale_log2, bias));
    l_state += a + b;
    p[i / 4].u[i % 4] = pack_bf16(a, b);
  };
  auto value_frag = [&](int at, int c, int dt) {   // 16 keys, 32 dims
    union { s16x4_t h[2]; bf16x8_t v; } vf;
#pragma unroll
    for (int x = 0; x < 2; ++x)
      vf.h[x] = read_transposed((lds_s16x4_t*)(v_lane[dt] + (at + (2 * c + x) * 8 * HD * 2)));
    return vf.v;
  };
  auto values = [&](const Probs (&p)[4], int buf) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(value_frag(buf * BYTES, c, dt), p[c].v,
                                                          acc[dt], 0, 0, 0);
  };

  int ids[PASS];         // block ids of the tile after the next to be asked for
  Place places[PASS];    // of the values that are asked for next
  if constexpr (TURNS) {
    // Two waves of a SIMD take turns: while one's probabilities are made, the other multiplies.
    // Both run the same program, waves 4 to 7 a barrier later: with barriers counted from the
    // first scores on, tile t's probabilities lie behind barrier 2 t + 1 (late: + 2), its values
    // and the next one's scores behind 2 t + 2 (+ 3).
    f32x16_t s[2];
    Probs p[4];
    const bool late = wave >= 4;
    auto turn = [&] {
      __builtin_amdgcn_sched_barrier(0);
      block_meet();
      __builtin_amdgcn_sched_barrier(0);
    };
    // Fragments are read a batch ahead, behind the first products of the batch before (the
    // compiler waits for all reads that are on their way, wherever it waits), the first batch
    // ahead of the barrier.
    constexpr int COUNT = HD / 8, BATCH = 4;   // products of values, of scores
    bf16x8_t kf[2 * BATCH], vf[2 * BATCH];
    auto fetch = [&](auto at, int g, bool keys) {
      constexpr int k_buf = (at + 1) % 3 * BYTES, v_buf = at * BYTES;
      if (keys) kf[g % (2 * BATCH)] = key_frag(k_buf, g);
      vf[g % (2 * BATCH)] = value_frag(v_buf, g / DT, g % DT);
    };
    auto multiply = [&](auto at, auto more, auto between) {
#pragma unroll
      for (int g = 0; g < COUNT; ++g) {
        if constexpr (more)
          s[g & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              kf[g % (2 * BATCH)], qf[g >> 1], g < 2 ? f32x16_t{} : s[g & 1], 0, 0, 0);
        acc[g % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[g % (2 * BATCH)], p[g / DT].v,
                                                              acc[g % DT], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (g % BATCH < 2 && g / BATCH + 1 < COUNT / BATCH) {
          fetch(at, (g / BATCH + 1) * BATCH + g % BATCH * 2, more);
          fetch(at, (g / BATCH + 1) * BATCH + g % BATCH * 2 + 1, more);
        }
        if (g == 2) between();
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // Behind barrier 2 u + 2 tile u + 3 of keys and u + 2 of values: their places were last read
    // ahead of it, in the late waves' products of tile u - 1.  They have landed ahead of barrier
    // 2 u + 4 and are first read behind 2 u + 5.
    auto plan = [&](Place (&ahead)[PASS], int u) {
      if (EVEN || u + 3 < n) places_of(ahead, ids, u + 3);
      if (EVEN || u + 4 < n) ids_of(ids, u + 4);
    };
    auto ask = [&](int u, auto at, Place (&ahead)[PASS]) {
      if constexpr (!EVEN) plan(ahead, u);
      if (u + 2 < n) issue(v_at, places, lds_all + (3 + (at + 2) % 3) * BYTES, vr, v_swz);
      if (u + 3 < n) issue(k_at, ahead, lds_all + at * BYTES, kr, k_swz);
    };
    auto landed = [&](int u, auto at) {
      if constexpr (FP8) {
        if (u + 2 < n) unpack(lds_all + (3 + (at + 2) % 3) * BYTES, vr, v_swz);
        if (u + 3 < n) unpack(lds_all + at * BYTES, kr, k_swz);
        __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0), lgkmcnt(0)
      } else {
        __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
      }
    };
    auto step = [&](int t, auto at) {   // at: t % 3
      Place ahead[PASS];
      if constexpr (EVEN) plan(ahead, t);   // where all waves come by: the scalar unit's
      turn();
      if (late) ask(t, at, ahead);
      const bool active = t * kTile <= wave_max;   // wave-uniform: the matrix unit wants all lanes
      if (active) {
        follow(s, t * kTile);
        bias = m_state == -FLT_MAX ? 0.f : -m_state * scale_log2;
#pragma unroll
        for (int i = 0; i < 16; ++i) weigh(s, p, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < BATCH; ++g) fetch(at, g, true);
      }
      if (!late && t > 0) landed(t - 1, std::integral_constant<int, (at + 2) % 3>{});
      turn();
      auto between = [&] {
        if (!late) ask(t, at, ahead);
      };
      if (active) {
        __builtin_amdgcn_s_setprio(1);
        if (t + 1 < n && (t + 1) * kTile <= wave_max)
          multiply(at, std::true_type{}, between);
        else
          multiply(at, std::false_type{}, between);
        __builtin_amdgcn_s_setprio(0);
      } else {
        between();
      }
      if (late) landed(t, at);
#pragma unroll
      for (int ps = 0; ps < PASS; ++ps) places[ps] = ahead[ps];
    };
    if (n > 0) {
      auto first_keys = [&](int t) {
        issue(k_at, places, lds_all + t * BYTES, kr, k_swz);
        if constexpr (FP8) unpack(lds_all + t * BYTES, kr, k_swz);
      };
      auto first_values = [&](int t) {
        issue(v_at, places, lds_all + (3 + t) * BYTES, vr, v_swz);
        if constexpr (FP8) unpack(lds_all + (3 + t) * BYTES, vr, v_swz);
      };
      ids_of(ids, 0);
      places_of(places, ids, 0);
      ids_of(ids, 1);
      first_keys(0);
      first_values(0);
      if (n > 1) {
        places_of(places, ids, 1);
        ids_of(ids, 2);
        first_keys(1);
        first_values(1);
        if (n > 2) {
          places_of(places, ids, 2);
          first_keys(2);
        }
        ids_of(ids, 3);
      }
      meet();
      if (late) turn();
      if (0 <= wave_max) scores(s, 0, [](int) {});
      for (int t = 0; t < n; t += 3) {
        step(t, std::integral_constant<int, 0>{});
        if (t + 1 < n) step(t + 1, std::integral_constant<int, 1>{});
        if (t + 2 < n) step(t + 2, std::integral_constant<int, 2>{});
      }
      if (!late) turn();
    }
  } else {
    f32x16_t s0[2], s1[2];
    auto step = [&](int t, f32x16_t (&now)[2], f32x16_t (&next)[2], int buf) {
      meet();
      const bool more_k = t + 2 < n, more_v = t + 1 < n;
      if constexpr (EVEN) {
        Place ahead[PASS];
        places_of(ahead, ids, t + 2);
        if (more_v) issue(v_at, places, v_lds[buf ^ 1], vr, v_swz);
        if (more_k) issue(k_at, ahead, k_lds[buf], kr, k_swz);
        ids_of(ids, t + 3);
#pragma unroll
        for (int ps = 0; ps < PASS; ++ps) places[ps] = ahead[ps];
      } else {
        if (more_v) issue(v_at, places, v_lds[buf ^ 1], vr, v_swz);
        if (more_k) {
          places_of(places, ids, t + 2);
          issue(k_at, places, k_lds[buf], kr, k_swz);
          if (t + 3 < n) ids_of(ids, t + 3);
        }
      }
      // wave-uniform: the matrix unit wants all lanes
      if (t * kTile <= wave_max) {
        Probs p[4];
        follow(now, t * kTile);
        bias = m_state == -FLT_MAX ? 0.f : -m_state * scale_log2;
        auto work = [&](int i) { weigh(now, p, i); };
        if (more_v && (t + 1) * kTile <= wave_max) {
          scores(next, (buf ^ 1) * BYTES, work);
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i) work(i);
        }
        values(p, buf);
      }
      if constexpr (FP8) {
        if (more_v) unpack(v_lds[buf ^ 1], vr, v_swz);
        if (more_k) unpack(k_lds[buf], kr, k_swz);
      }
    };
    if (n > 0) {
      ids_of(ids, 0);
      places_of(places, ids, 0);
      issue(k_at, places, k_lds[0], kr, k_swz);
      issue(v_at, places, v_lds[0], vr, v_swz);
      if constexpr (FP8) {
        unpack(k_lds[0], kr, k_swz);
        unpack(v_lds[0], vr, v_swz);
      }
      if (n > 1) {
        ids_of(ids, 1);
        places_of(places, ids, 1);
        issue(k_at, places, k_lds[1], kr, k_swz);
        if constexpr (FP8) unpack(k_lds[1], kr, k_swz);
        if (EVEN || n > 2) ids_of(ids, 2);
      }
      meet();
      if (0 <= wave_max) scores(s0, 0, [](int) {});
      for (int t = 0; t < n; t += 2) {
        step(t, s0, s1, 0);
        if (t + 1 < n) step(t + 1, s1, s0, 1);
      }
    }
  }

  l_state += __shfl_xor(l_state, 32, 64);
  const bool mine = token0 + col < q_len;
  const long row = (long)(q_start + token) * nheads + head;
  if (per < tiles) {
    if (!mine) return;
    const long at = blockIdx.z % parts * ((long)query_start_loc[gridDim.y] * nheads) + row;
    float* o = part_acc + at * HD + half * 4;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<f32x4_t*>(o + dt * 32 + r * 2) =
            f32x4_t{acc[dt][r], acc[dt][r + 1], acc[dt][r + 2], acc[dt][r + 3]};
    if (half == 0) {
      part_ml[at * 2] = m_state == -FLT_MAX ? -FLT_MAX : m_state * scale_log2;
      part_ml[at * 2 + 1] = l_state;
    }
    return;
  }
  const float inv = l_state > 0.f ? 1.f / l_state : 0.f;
  // the halves swap, so that a lane has eight neighbours
  __hip_bfloat16* o = out + row * HD + half * 8;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; r += 8) {
      u32x4_t w;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int at = r + 2 * i;
        const auto both = __builtin_amdgcn_permlane32_swap(
            pack_bf16(acc[dt][at] * inv, acc[dt][at + 1] * inv),
            pack_bf16(acc[dt][at + 4] * inv, acc[dt][at + 5] * inv), false, false);
        w[i] = both[0];
        w[i + 2] = both[1];
      }
      if (mine) *reinterpret_cast<u32x4_t*>(o + dt * 32 + r * 2) = w;
    }
}

// Tokens whose keys were cut: out = sum_p f_p acc_p / sum_p f_p l_p.  grid (tokens of the
// longest prompt, sequences, heads / 4), a wave a head; parts <= 16.
template <int HD>
__global__ __launch_bounds__(256) void prefill_tile_merge_kernel(
    __hip_bfloat16* __restrict__ out, const float* __restrict__ part_acc,
    const float* __restrict__ part_ml, const int* __restrict__ query_start_loc,
    const int* __restrict__ seq_lens, const int nheads, const int tokens, const int parts) {
  const int seq = blockIdx.y, token = blockIdx.x;
  const int head = blockIdx.z * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int q_start = query_start_loc[seq], q_len = query_start_loc[seq + 1] - q_start;
  if (token >= q_len || head >= nheads) return;
  const int seq_len = seq_lens[seq], past = seq_len - q_len;
  const int keys = min(seq_len, past + min((token / tokens + 1) * tokens, q_len));
  const int tiles = (keys + kTile - 1) / kTile, per = tiles_per_part(tiles, parts);
  if (per >= tiles) return;
  const int used = (tiles + per - 1) / per;
  const long rows = (long)query_start_loc[gridDim.y] * nheads;
  const long row = (long)(q_start + token) * nheads + head;
  const float* ml = part_ml + (min(lane, used - 1) * rows + row) * 2;
  const float m = lane < used ? ml[0] : -FLT_MAX, l = lane < used ? ml[1] : 0.f;
  constexpr int V = HD / 64;
  const float* acc = part_acc + row * HD + lane * V;
  float a[V] = {};
  const float top = wave_reduce_max(m);
  const float f = lane < used ? __builtin_amdgcn_exp2f(m - top) : 0.f;
  const float sum = wave_reduce_sum(f * l);
  for (int p0 = 0; p0 < used; p0 += 4) {   // four loads on their way at a time
    float v[4][V];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < V; ++j) v[i][j] = acc[min(p0 + i, used - 1) * rows * HD + j];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (p0 + i < used)
#pragma unroll
        for (int j = 0; j < V; ++j) a[j] += __shfl(f, p0 + i, 64) * v[i][j];
  }
  const float inv = sum > 0.f ? 1.f / sum : 0.f;
#pragma unroll
  for (int j = 0; j < V; ++j) out[row * HD + lane * V + j] = __float2bfloat16(a[j] * inv);
}

struct Cut {
  int waves, heads, tokens, parts;   // of a workgroup; workgroups a tile's keys are cut over
};

void shape(Cut& c, int waves, int group) {
  c.waves = c.heads = waves;
  while (group % c.heads) c.heads /= 2;
  c.tokens = waves / c.heads * 32;
}

long blocks_of(const Cut& c, int nseq, int nheads, int max_query_len) {
  const long n = (long)nheads / c.heads * nseq * ((max_query_len + c.tokens - 1) / c.tokens);
  return n > 0 ? n : 1;
}

// Eight waves share every tile of keys where their workgroups, with the keys cut into parts
// where there are few, fill more than half the chip; else four do, two such workgroups a
// CU.  Measured, heads 32/8 of 128 (us, waves/parts): 3500 tokens of 7 prompts after 700
// each 8/1 87, 4/1 88, 8/2 133; 512 after 5000 8/1 167, 4/1 146, 8/2 99, 8/4 65, 4/4 69, 8/8
// 77; 1000 after 3000 8/1 130, 8/2 87, 8/4 91; 64 after 6000 4/1 157, 4/8 34, 4/16 29, 8/16
// 33; 4 of 100 after 1000 8/1 41, 4/1 36, 4/2 34; 4 of 50 after 500 (9 tiles) 4/1 21, 4/2 26;
// one of 300 8/1 17, 4/1 14.5.
//
// With few query heads a key head the waves take tokens, and half as many waves go where the
// longest prompt leaves half of them idle: heads 12/12 of 64 (us, 8 | 4 | 2 waves): 64 prompts
// of 17 tokens 13.1 | 9.1 | 6.7, 300 of 9 | 29.6 | 18.3.  Idle waves still stage keys: with
// long contexts all eight are worth it (16/16 heads of 128, 64 tokens after 4000 22.6 | 24.2),
// two do for a few tiles only (16/8, 100 of 5 after 500 | 55 | 66), and e4m3 keys, which are
// widened, take more (16/16, 16 of 128 11.5 | 12.6, 8 of 30 | 7.2 | 8.5).
Cut waves_of(bool fp8, int nseq, int nheads, int kvh, int max_query_len, int max_keys) {
  const int group = nheads / kvh, most = max_keys / (kTile * 6);
  Cut c{};
  for (c.waves = 8;; c.waves /= 2) {
    shape(c, c.waves, group);
    const long blocks = blocks_of(c, nseq, nheads, max_query_len);
    const long fit = 256 * 8 / c.waves / blocks;
    c.parts = fit < 16 ? (int)fit : 16;
    if (c.parts > most) c.parts = most;
    if (c.parts < 1) c.parts = 1;
    const bool idle = c.tokens > 32 && max_keys <= 8 * kTile &&
                      max_query_len <= c.tokens / (fp8 ? 8 : 2);
    const bool least = c.waves == (fp8 || max_keys > 2 * kTile ? 4 : 2);
    if (least || (!idle && (c.waves == 4 || blocks * c.parts > 128))) return c;
  }
}

// Four or eight query heads a key head: the parts again, and for bf16 keys four waves instead of
// eight, by what a launch takes, us: its start, the longest chain of tiles, and for parts their launch,
// their sums written and read.  Fitted to some 1000 times (heads 32/8 of 128 and 64, 64/8 of 128; one to
// sixteen prompts of 2 to 8192 tokens, after none to 6000).
//  - Parts pay for their sums only where tokens are few: one prompt of 1000 in 8 waves, 2 parts 37.8, 1
//    part 30.9, by 4 waves 29.0; heads of 64 29.0 | 20.3, e4m3 40.0 | 33.3 by 8; after 1000 tokens, heads of 64, 40.9 | 35.4; 64/8
//    heads, 512 after 1000 46.7 | 41.6; but 1000 after 3000 78.6 | 96.  Fewer parts than fill the chip,
//    but some, are never faster: what few tokens leave stays in the caches (10 | 8 parts, e4m3, 2 prompts of
//    64 after 4000 33.8 | 36.1, 64/8 heads, 64 after 4000 32.1 | 33.7; 15 | 12, 30 after 6000 26.2 | 26.6).
//  - Uncut, four waves end a workgroup's last tiles sooner, where they are one a CU, or, where many keys
//    are the prompts' own, two and their tiles few (heads of 64: up to three): 8 | 4 waves, 32/8 heads
//    of 128, 2 prompts of 1000 33.3 | 32.4, 8 of 256 16.6 | 15.1; of 64, one of 2000 40.4 | 36.6, 4 of 500
//    after 700 28.8 | 26.4; past that 7 of 500 after 700 67.6 | 70.1, one of 4000 132 | 145; 64/8 heads,
//    8 of 128 after 600 31.3 | 34.1, one of 2000 73.8 | 79.3; e4m3, 2 prompts of 1000 37.0 | 37.6.
//  - Where lanes find their rows (not `even`: blocks of 24) a tile takes longer, by four waves more so: four
//    where they are the faster by times of their own (8 | 4 waves, 32/8 heads of 128, one of 512 23.1 | 21.7, 8
//    of 256 18.3 | 17.3, but one of 1000 36.8 | 37.4, 2 of 1000 38.8 | 39.9, 1000 after 500 in 2 parts 48.3 |
//    53.4; of 64, one of 1000 25.9 | 24.6, 700 after 700 33.9 | 32.0, but 512 after 1000 in 3 parts 29.4 |
//    34.1, 3 of 1000 27.2 | 28.4, 64/8 heads, 1500 after 1500 93 | 104).
Cut cut_of(bool fp8, bool even, int nseq, int nheads, int kvh, int head_dim, int max_query_len,
           int max_keys) {
  Cut c = waves_of(fp8, nseq, nheads, kvh, max_query_len, max_keys);
  const int group = nheads / kvh;
  if (group % 4 != 0 || c.waves < 4) return c;
  const bool wide = head_dim == 128;
  const int tiles = (max_keys + kTile - 1) / kTile, least = kMinTiles;
  const double mb = 8e-6 * nseq * max_query_len * nheads * head_dim;   // of a part, there and back
  const bool lanes = !even && !fp8 && c.waves == 8;   // (e4m3 keys stay with eight waves or four)
  auto us = [&](int waves, int parts) {
    const int per = parts == 1 || tiles <= least ? tiles : std::max(least, (tiles + parts - 1) / parts);
    const double start = fp8    ? (waves == 8 ? 7.0 : 4.5)
                         : wide ? (waves == 8 ? 8.1 : 6.1) : (waves == 8 ? 5.7 : 4.6);
    const double tile = fp8             ? (waves == 8 ? 1.65 : 1.83)
                        : lanes && wide ? (waves == 8 ? 1.8 : 1.95)
                        : lanes         ? (waves == 8 ? 1.25 : 1.22)
                        : wide          ? (waves == 8 ? 1.44 : 1.42) : (waves == 8 ? 1.3 : 0.95);
    return start + tile * per +
           (parts > 1 ? 3.5 + 0.3 * parts + (wide ? 0.21 : 0.35) * mb * parts : 0.0);
  };
  const long fit = 256 * 8 / c.waves / blocks_of(c, nseq, nheads, max_query_len);
  const int most = max_keys / (kTile * least), filling = std::max(2, c.parts);
  c.parts = 1;
  for (int p = filling; p <= 16 && p <= fit && p <= most; ++p)
    if (us(c.waves, p) < us(c.waves, c.parts)) c.parts = p;
  if (c.waves == 8 && !fp8) {
    Cut four{};
    shape(four, 4, group);
    four.parts = 1;
    const long blocks = blocks_of(four, nseq, nheads, max_query_len);
    const bool own = 2L * max_keys <= 5L * max_query_len;
    const bool short_chain = own && (wide ? blocks <= 512 && tiles <= 16 : blocks <= 768);
    if (lanes          ? blocks <= (own || c.parts > 1 ? 512 : 256) && us(4, 1) < us(8, c.parts)
        : c.parts == 1 ? blocks <= 256 || short_chain
                       : blocks <= 512 && us(4, 1) < 0.95 * us(8, c.parts))
      c = four;
  }
  return c;
}

// Whether a wave's loads lie inside cache blocks and are found by the scalar unit: see the kernel.
bool even_blocks(int block_size, int kvh, int head_dim, int bytes) {
  return (block_size & (block_size - 1)) == 0 && block_size % (1024 / (head_dim * bytes)) == 0 &&
         (long)kvh * head_dim * bytes < 1 << 24;
}

template <int HD, typename CT>
void launch(__hip_bfloat16* out, float* part_acc, float* part_ml, const __hip_bfloat16* q,
            const CT* kc, const CT* vc, const int* bt, const int* qsl, const int* sl,
            float scale, int nseq, int nheads, int kvh, int block_size, int max_blocks,
            int max_query_len, const Cut& c, hipStream_t stream) {
  const int shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz(block_size) : -1;
  const int tiles = (max_query_len + c.tokens - 1) / c.tokens;
  auto go = [&](auto kernel, bool turns) {
    hipLaunchKernelGGL(kernel, dim3(nheads / c.heads, nseq, tiles * c.parts),
                       dim3(c.waves * 64), turns ? 0 : 4 * kTile * HD * 2, stream, out, q, kc, vc, bt, qsl,
                       sl, scale * kLog2e, nheads, kvh, c.heads, block_size, shift, max_blocks,
                       c.parts, part_acc, part_ml);
  };
  const bool even = even_blocks(block_size, kvh, HD, sizeof(CT));
#define GO(NW, EVEN) go(paged_prefill_tile_kernel<HD, CT, NW, EVEN>, kTurns<HD, CT, NW, EVEN>)
  if (c.waves == 8 && even) GO(8, true);
  else if (c.waves == 8) GO(8, false);
  else if (c.waves == 4 && even) GO(4, true);
  else if (c.waves == 4) GO(4, false);
  else if (even) GO(2, true);
  else GO(2, false);
#undef GO
  if (c.parts > 1)
    hipLaunchKernelGGL((prefill_tile_merge_kernel<HD>), dim3(max_query_len, nseq, (nheads + 3) / 4),
                       dim3(256), 0, stream, out, part_acc, part_ml, qsl, sl, nheads, c.tokens, c.parts);
}

}  // namespace

// Waves of a workgroup << 8 | workgroups that a prompt's keys may be cut over (a function of shapes
// only): 1, or the launch needs part_acc [parts, tokens, nheads, head_dim] and part_ml [parts, tokens,
// nheads, 2].
int prefill_tile_plan(bool fp8, int block_size, int nseq, int nheads, int kvh, int head_dim,
                      int max_query_len, int max_keys) {
  const Cut c = cut_of(fp8, even_blocks(block_size, kvh, head_dim, fp8 ? 1 : 2), nseq, nheads, kvh,
                       head_dim, max_query_len, max_keys);
  return c.waves << 8 | c.parts;
}

void launch_paged_prefill_tile(__hip_bfloat16* out, float* part_acc, float* part_ml,
                               const __hip_bfloat16* q, const __hip_bfloat16* kc,
                               const __hip_bfloat16* vc, const int* bt, const int* qsl,
                               const int* sl, float scale, int nseq, int nheads, int kvh,
                               int head_dim, int block_size, int max_blocks, int max_query_len,
                               int max_keys, hipStream_t stream) {
  const Cut c = cut_of(false, even_blocks(block_size, kvh, head_dim, 2), nseq, nheads, kvh, head_dim,
                       max_query_len, max_keys);
  auto go = [&](auto launch) {
    launch(out, part_acc, part_ml, q, kc, vc, bt, qsl, sl, scale, nseq, nheads, kvh, block_size,
           max_blocks, max_query_len, c, stream);
  };
  if (head_dim == 128) go(launch<128, __hip_bfloat16>);
  else go(launch<64, __hip_bfloat16>);
}

// heads of 128
void launch_paged_prefill_tile_fp8(__hip_bfloat16* out, float* part_acc, float* part_ml,
                                   const __hip_bfloat16* q, const unsigned char* kc,
                                   const unsigned char* vc, const int* bt, const int* qsl,
                                   const int* sl, float scale, int nseq, int nheads, int kvh,
                                   int block_size, int max_blocks, int max_query_len,
                                   int max_keys, hipStream_t stream) {
  launch<128, unsigned char>(out, part_acc, part_ml, q, kc, vc, bt, qsl, sl, scale, nseq, nheads,
                             kvh, block_size, max_blocks, max_query_len,
                             cut_of(true, even_blocks(block_size, kvh, 128, 1), nseq, nheads, kvh,
                                    128, max_query_len, max_keys), stream);
}
