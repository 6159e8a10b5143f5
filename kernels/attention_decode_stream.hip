// Paged decode attention, one query row per sequence: bf16 or e4m3 cache, heads of
// 64 or 128, up to 8 query heads per key head.
//
// Bound by the cache's bytes.  Every wave walks 32-key tiles: keys and values are
// loaded as whole rows (a tile of both in registers while the one before is worked
// on, its block ids a tile earlier still), keys, then values, go through the wave's
// own LDS tile.  v_mfma_f32_16x16x32_bf16 takes S^T = K Q^T, so a lane keeps one
// query's statistics and accumulators and no shuffle rescales them; the two 16-key
// score tiles take the second product's slots in the order the score layout has
// them, so probabilities are packed where they are, and the values come back
// transposed (ds_read_b64_tr_b16), swizzled so that neither way has bank conflicts.
// The rows are read once: loads that leave no trace in the caches (nontemporal).
//
// The keys of a sequence are cut over up to npart workgroups (a pure function of
// shapes, so that a captured launch stays valid) of at least four tiles each, the
// four waves merge in LDS, and only a sequence that was cut goes through the merge
// kernel.  Of many short sequences a wave takes a key head by itself (alone_tiles): the
// lengths say so on the device, so that a captured launch serves both.
//
// Measured (MI355X, 32/8 heads of 128, two layers with their cache writes): 512
// sequences of ~520 keys, bf16: 794 -> 361 us (2.8 -> 6.1 TB/s; a plain read
// reaches 6.3); 41 of ~4800 keys, e4m3: 1365 -> 165 us (the former kernel ran 328
// workgroups there).  On the way: three workgroups a CU instead of two spill, 427;
// cached loads, 407; keys loaded straight into the operand's layout, 398.

#include "common.h"
#include <float.h>

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

namespace {

constexpr int kTile = 32;    // keys per wave and step
constexpr int kWaves = 4;
constexpr int kMinTiles = kWaves;   // a workgroup's share is no smaller
constexpr float kLog2e = 1.4426950408889634f;

DEVINLINE unsigned pack_bf16(float a, float b) {
  unsigned r;
  asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// tiles of a sequence that one workgroup takes, a multiple of the waves
DEVINLINE int tiles_per_part(int tiles, int npart) {
  const int per = (tiles + npart - 1) / npart;
  return max(kMinTiles, (per + kWaves - 1) / kWaves * kWaves);
}

// A load that is asked for where it stands: the compiler would move it behind a branch
template <typename T> DEVINLINE T load_here(const T* at) {
  return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// What a wave does with its tiles of 32 keys of one key head.
template <int HD, typename CT> struct Walk {
  static constexpr bool FP8 = sizeof(CT) == 1;
  static constexpr int KS = HD / 32;              // contraction steps of a score tile
  static constexpr int DT = HD / 16;              // 16-wide tiles of the result
  static constexpr int PER = 16 / sizeof(CT);     // elements of a 16-byte load
  static constexpr int LPR = HD / PER;            // lanes per value row
  static constexpr int RPP = 64 / LPR;            // value rows per pass
  static constexpr int VP = kTile / RPP;          // passes

  char* lds;                                 // the wave's tile
  int lane, col, quad;
  bf16x8_t qf[KS];
  u32x4_t kr[VP], vr[VP];                    // the tile that is on its way
  float m_state, l_state;                    // of query `col`; l: this lane's keys
  f32x4_t acc[DT];

  DEVINLINE void begin() {
    m_state = -FLT_MAX;
    l_state = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4_t{};
  }
  // queries of `group` heads from `from` on
  DEVINLINE void ask_queries(bf16x8_t (&to)[KS], const __hip_bfloat16* from, int group) const {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      to[ks] = bf16x8_t{};
      if (col < group)
        to[ks] = *reinterpret_cast<const bf16x8_t*>(from + col * HD + ks * 32 + quad * 8);
    }
  }
  // slot: cache row of the tile's key lane % 32
  DEVINLINE void issue(const CT* k_cache, const CT* v_cache, int slot, int kv_head,
                       long row_elems) {
    long at[VP];
#pragma unroll
    for (int ps = 0; ps < VP; ++ps)
      at[ps] = __shfl(slot, ps * RPP + lane / LPR, 64) * row_elems + kv_head * HD +
               (lane % LPR) * PER;
#pragma unroll
    for (int ps = 0; ps < VP; ++ps)
      kr[ps] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(k_cache + at[ps]));
#pragma unroll
    for (int ps = 0; ps < VP; ++ps)
      vr[ps] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(v_cache + at[ps]));
  }
  // 16-byte chunk c of row r lies at chunk c ^ swizzle(r): a pair of chunks stays a
  // pair, the 16 rows of a transposed read cover all banks twice, and eight rows'
  // equal chunks lie in different banks
  static DEVINLINE int swizzle(int r) { return HD == 128 ? (r & 7) * 2 : ((r >> 1) & 3) * 2; }
  DEVINLINE void stage(const u32x4_t (&from)[VP]) const {
#pragma unroll
    for (int ps = 0; ps < VP; ++ps) {
      const int r = ps * RPP + lane / LPR;
      char* row = lds + r * HD * 2;
      if constexpr (FP8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          u32x2_vec_t u;
          u[0] = from[ps][2 * h];
          u[1] = from[ps][2 * h + 1];
          *reinterpret_cast<bf16x8_vec_t*>(
              row + (((lane % LPR) * 2 + h) ^ swizzle(r)) * 16) = fp8x8_to_bf16x8(u);
        }
      } else {
        *reinterpret_cast<u32x4_t*>(row + ((lane % LPR) ^ swizzle(r)) * 16) = from[ps];
      }
    }
    // other lanes of this wave read it: LDS keeps a wave's order, the compiler has to
    asm volatile("" ::: "memory");
  }
  // The tile on its way, of keys key0 .. key0 + 31; `next` asks for the one after it.
  template <typename Next>
  DEVINLINE void work(const int key0, const int seq_len, const float scale_log2, Next next) {
    f32x4_t s[2] = {f32x4_t{}, f32x4_t{}};
    stage(kr);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const int r = rt * 16 + col;
        const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(
            lds + r * HD * 2 + ((ks * 4 + quad) ^ swizzle(r)) * 16);
        s[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[ks], s[rt], 0, 0, 0);
      }
    asm volatile("" ::: "memory");
    stage(vr);
    next();

    // ---- softmax: lane has keys rt*16 + quad*4 + r of query col ----------
    const int base = key0 + quad * 4;
    float big = -FLT_MAX;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = s[rt][r] * scale_log2;
        if (base + rt * 16 + r >= seq_len) v = -FLT_MAX;
        s[rt][r] = v;
        big = fmaxf(big, v);
      }
    big = fmaxf(big, __shfl_xor(big, 16, 64));
    big = fmaxf(big, __shfl_xor(big, 32, 64));
    const float m_new = fmaxf(m_state, big);
    if (!__all(m_new == m_state)) {
      const float f = __builtin_amdgcn_exp2f(m_state - m_new);
      l_state *= f;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[dt][r] *= f;
      m_state = m_new;
    }
    union { unsigned u[4]; bf16x8_t v; } p;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      float e[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        e[r] = s[rt][r] == -FLT_MAX ? 0.f : __builtin_amdgcn_exp2f(s[rt][r] - m_state);
        l_state += e[r];
      }
      p.u[2 * rt] = pack_bf16(e[0], e[1]);
      p.u[2 * rt + 1] = pack_bf16(e[2], e[3]);
    }

    // ---- O^T += V^T P^T, values read back transposed ---------------------
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      union { s16x4_t h[2]; bf16x8_t v; } vf;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const int r = rt * 16 + quad * 4 + (col >> 2);
        char* at = lds + r * HD * 2 + ((dt * 2 + ((col & 3) >> 1)) ^ swizzle(r)) * 16 +
                   (col & 1) * 8;
        vf.h[rt] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)at);
      }
      acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, p.v, acc[dt], 0, 0, 0);
    }
    asm volatile("" ::: "memory");
  }
  // l of all of the tiles' keys
  DEVINLINE void end() {
    l_state += __shfl_xor(l_state, 16, 64);
    l_state += __shfl_xor(l_state, 32, 64);
  }
};

// CUT: npart > 1.  ALONE: some sequences' key heads may be a wave's each (as a question of every launch
// it took 0.1 to 0.4 us of small batches': 20 x 60 keys 6.87 | 7.24)
template <int HD, typename CT, bool CUT, bool ALONE>
__global__ __launch_bounds__(256, 2) void paged_decode_stream_kernel(
    __hip_bfloat16* __restrict__ out,       // [nseq, nheads, HD]
    float* __restrict__ part_acc,           // [nseq, nheads, npart, HD] (npart > 1)
    float* __restrict__ part_ml,            // [nseq, nheads, npart, 2]  (npart > 1)
    const __hip_bfloat16* __restrict__ q,   // [nseq, nheads, HD]
    const CT* __restrict__ k_cache,         // [blocks, block_size, kvh, HD]
    const CT* __restrict__ v_cache,
    const int* __restrict__ block_tables,   // [nseq, max_blocks]
    const int* __restrict__ seq_lens,       // [nseq]
    const float scale_log2, const int nheads, const int kvh, const int group,
    const int block_size, const int block_shift, const int max_blocks,
    const int alone_tiles) {   // see the rule of that name
  using W = Walk<HD, CT>;
  const int seq = blockIdx.x, part = blockIdx.z;
  int kv_head = blockIdx.y;
  const int npart = gridDim.z;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int* table = block_tables + (long)seq * max_blocks;

  // Where a sequence is cut, and so the launch short, and a workgroup's first tile does not depend on
  // the length, block ids are asked for beside it (with the merge's loads, us: one sequence of 230 keys
  // of 64 6.8 -> 6.5, of 700 keys of 128 8.4 -> 8.0, of 8000 in e4m3 16.8 -> 15.1).  Past the end of the
  // sequence, but not of its table, they may be anything.
  const int most = max_blocks * block_size;
  const bool early = CUT && (part == 0 || most <= npart * (kMinTiles * kTile));
  auto page_of = [&](int pos) { return block_shift >= 0 ? pos >> block_shift : pos / block_size; };
  const int pos0 = (part * kMinTiles + wave) * kTile + (lane & 31);
  int entry0 = 0;
  if (early) entry0 = load_here(table + page_of(min(pos0, most - 1)));
  const int seq_len = seq_lens[seq];
  const int tiles = (seq_len + kTile - 1) / kTile;
  const int tpp = tiles_per_part(tiles, npart);
  const int lo = part * tpp;
  // a sequence without keys (padding) still gets its zeros from part 0
  if (lo >= tiles && part > 0) return;
  const int hi = min(lo + tpp, tiles);
  // Few keys: a wave takes a key head by itself, every fourth workgroup four of them.
  const bool alone = ALONE && tiles <= alone_tiles;
  if (alone) {
    if (kv_head % kWaves != 0) return;
    kv_head += wave;
  }

  const int head0 = kv_head * group;
  const long row_elems = (long)kvh * HD;

  __shared__ __align__(16) __hip_bfloat16 tile_all[kWaves][kTile * HD];
  __shared__ float ml_all[kWaves][2][16];
  W walk;
  walk.lds = reinterpret_cast<char*>(tile_all[wave]);
  walk.lane = lane;
  walk.col = lane & 15;
  walk.quad = lane >> 4;
  const int col = walk.col, quad = walk.quad;
  walk.ask_queries(walk.qf, q + ((long)seq * nheads + head0) * HD, group);

  // cache row of key (tile * 32 + lane % 32); past the end: of the last key
  auto slot_of = [&](int tile) {
    const int pos = min(tile * kTile + (lane & 31), seq_len - 1);
    const int page = page_of(pos);
    return table[page] * block_size + (pos - page * block_size);
  };
  walk.begin();

  int t = alone ? 0 : lo + wave, slot_next = 0;
  const int stride = alone ? 1 : kWaves;
  if (t < hi) {
    int slot;
    if (early && !alone) {   // past the end: of the tile's first key
      slot = (unsigned)entry0 * block_size + (pos0 - page_of(pos0) * block_size);
      const int begin = __shfl(slot, 0, 64);
      if (pos0 >= seq_len) slot = begin;
    } else {
      slot = slot_of(t);
    }
    walk.issue(k_cache, v_cache, slot, kv_head, row_elems);
    if (t + stride < hi) slot_next = slot_of(t + stride);
  }
  for (; t < hi; t += stride)
    walk.work(t * kTile, seq_len, scale_log2, [&] {
      if (t + stride < hi) {
        walk.issue(k_cache, v_cache, slot_next, kv_head, row_elems);
        if (t + 2 * stride < hi) slot_next = slot_of(t + 2 * stride);
      }
    });
  walk.end();
  if (alone) {
    if (col >= group) return;
    const float inv = walk.l_state > 0.f ? 1.f / walk.l_state : 0.f;
    __hip_bfloat16* o = out + ((long)seq * nheads + head0 + col) * HD + quad * 4;
#pragma unroll
    for (int dt = 0; dt < W::DT; ++dt)
      *reinterpret_cast<uint2*>(o + dt * 16) =
          uint2{pack_bf16(walk.acc[dt][0] * inv, walk.acc[dt][1] * inv),
                pack_bf16(walk.acc[dt][2] * inv, walk.acc[dt][3] * inv)};
    return;
  }

  // ---- the waves' results become one ---------------------------------------
  if (lane < 16) {
    ml_all[wave][0][lane] = walk.m_state;
    ml_all[wave][1][lane] = walk.l_state;
  }
  __syncthreads();
  float M = ml_all[0][0][col];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) M = fmaxf(M, ml_all[w][0][col]);
  const float f = __builtin_amdgcn_exp2f(walk.m_state - M);
  float* mine = reinterpret_cast<float*>(tile_all[wave]);   // [16][HD]
  static_assert(kTile * 2 >= 16 * 4, "a wave's tile holds its result");
  if (col < group) {
#pragma unroll
    for (int dt = 0; dt < W::DT; ++dt)
      *reinterpret_cast<f32x4_t*>(mine + col * HD + dt * 16 + quad * 4) = walk.acc[dt] * f;
  }
  __syncthreads();
  const bool whole = tpp >= tiles;
  for (int i = tid; i < group * HD; i += 256) {
    const int g = i / HD, d = i % HD;
    float top = ml_all[0][0][g];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) top = fmaxf(top, ml_all[w][0][g]);
    float a = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      a += reinterpret_cast<const float*>(tile_all[w])[i];
      l += ml_all[w][1][g] * __builtin_amdgcn_exp2f(ml_all[w][0][g] - top);
    }
    const long row = (long)seq * nheads + head0 + g;
    if (whole) {
      out[row * HD + d] = __float2bfloat16(a * (l > 0.f ? 1.f / l : 0.f));
    } else {
      part_acc[(row * npart + part) * HD + d] = a;
      if (d == 0) {
        part_ml[(row * npart + part) * 2] = top;
        part_ml[(row * npart + part) * 2 + 1] = l;
      }
    }
  }
}

// Sequences that were cut: out = sum_p f_p acc_p / sum_p f_p l_p.
template <int HD>
__global__ __launch_bounds__(HD) void decode_stream_merge_kernel(
    __hip_bfloat16* __restrict__ out, const float* __restrict__ part_acc,
    const float* __restrict__ part_ml, const int* __restrict__ seq_lens,
    const int nheads, const int npart) {
  const int seq = blockIdx.x, d = threadIdx.x;
  const long row = (long)seq * nheads + blockIdx.y;
  const int lane = d & 63;
  const float* ml = part_ml + row * npart * 2;
  const float* acc = part_acc + row * npart * HD + d;
  // For few rows all is asked for beside the length: parts that are not used hold anything, and are
  // not.  More rows would read in vain what their sequences, if whole, have not written (124 sequences
  // of 20 keys, 64 heads, two layers with their cache writes: 37.1 us, all asked for 40.4).
  const bool early = gridDim.x * gridDim.y <= 256;
  float m0 = 0.f, l0 = 0.f, v[8];   // eight loads on their way at a time
  auto ask = [&](int parts) {
    m0 = load_here(ml + 2 * min(lane, parts - 1));
    l0 = load_here(ml + 2 * min(lane, parts - 1) + 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = load_here(acc + (long)min(i, parts - 1) * HD);
  };
  if (early) ask(npart);
  const int tiles = (seq_lens[seq] + kTile - 1) / kTile;
  const int tpp = tiles_per_part(tiles, npart);
  if (tpp >= tiles) return;
  const int used = (tiles + tpp - 1) / tpp;   // <= npart <= 64
  if (!early) ask(used);
  const float m = lane < used ? m0 : -FLT_MAX;
  const float l = lane < used ? l0 : 0.f;
  const float M = wave_reduce_max(m);
  const float f = lane < used ? __builtin_amdgcn_exp2f(m - M) : 0.f;
  const float L = wave_reduce_sum(f * l);
  float a = 0.f;
  for (int p0 = 0;;) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (p0 + i < used) a += __shfl(f, p0 + i, 64) * v[i];
    p0 += 8;
    if (p0 >= used) break;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = acc[(long)min(p0 + i, used - 1) * HD];
  }
  out[row * HD + d] = __float2bfloat16(a * (L > 0.f ? 1.f / L : 0.f));
}

// Up to how many tiles a sequence's key heads are a wave's each instead of a workgroup's, -1: never.
// With a tile or two most waves of a workgroup have none, and what it takes is its chain of loads
// and the waves' meeting: worth it where the workgroups are more than are resident at a time (two or
// three a CU).  Two layers with their cache writes, us, a head a workgroup | up to 1, 2, 4, 6 tiles a head a
// wave; 32/8 heads of 128, sequences x mean keys: 453 x 34 75.8 | 68.1, 51.2, 51.1, 51.1 (e4m3 60.1 |
// 51.6, 39.1, 39.0, 38.7); 194 x 62 47.1 | 46.4, 43.3, 42.5, 42.4; 190 x 90 64.3 | 64.8, 64.8, 60.9, 69.0;
// 400 x 128 105.6 | 105.5, 104.8, 101.6, 98.9; 100 x 60 36.9 | 36.7, 35.3, 35.9, 35.9; 50 x 60 27.4 |
// 27.3, 29.7, 33.4, 33.5; 64 x 30 26.4 | 26.5, 31.6; 64/8 heads, 81 x 22 35.3 | 28.8, 30.6, 30.5; heads of
// 64, 512 x 50 48.5 | 48.1, 42.7, 39.8, 39.7.  (The workgroups that work first instead of every fourth:
// the same there, and 512 x 520 0.8 % slower.)
// What there is to win grows with the queries of a head, whose sums the waves would meet over, and shrinks
// with smaller tiles (heads of 64, e4m3), of which more workgroups are resident.  20 layers in turn, so many
// that no cache holds them, tables of 2048 keys; us of a launch, a head a workgroup | a wave, sequences x
// keys (up to), below the lines and past them: 32/8 heads of 64, 80 x 60 7.2 | 7.9, 192 x 120 in 4 tiles
// 9.8 | 10.5, 320 x 90 12.6 | 11.1; e4m3, 80 x 60 8.6 | 9.6, 128 x 60 11.9 | 10.2; one query a head, 32/32 of 128,
// 24 x 60 10.5 | 11.7, 48 x 180 22.3 | 25.7, 12/12 of 64, 64 x 60 6.7 | 9.1, 192 x 120 12.5 | 13.5.  With these lines
// none of 1352 such launches is 3 % slower than a head a workgroup, and the mean is 0.875 of it.
int alone_tiles(int nseq, int kvh, int group, int head_dim, bool fp8) {
  if (kvh % kWaves != 0) return -1;
  const long heads = (long)nseq * kvh;
  if (group < 4) return heads >= 3072 ? 4 : heads >= (head_dim == 64 ? 1344 : 2560) ? 2 : -1;
  if (head_dim == 64) return heads >= 2048 ? 4 : heads >= 1280 ? 2 : -1;
  return heads >= 1536 ? 4 : heads >= (fp8 ? 896 : 640) ? 2 : -1;
}

template <int HD, typename CT>
void launch(__hip_bfloat16* out, float* part_acc, float* part_ml, const __hip_bfloat16* q,
            const CT* kc, const CT* vc, const int* bt, const int* sl, float scale, int nseq,
            int nheads, int kvh, int block_size, int max_blocks, int npart,
            hipStream_t stream) {
  int shift = -1;
  if ((block_size & (block_size - 1)) == 0) shift = __builtin_ctz(block_size);
  // (a wave's results of a head by itself are stored by 8 bytes, a workgroup's one by one)
  const int alone = reinterpret_cast<uintptr_t>(out) % 8 == 0
                        ? alone_tiles(nseq, kvh, nheads / kvh, HD, sizeof(CT) == 1) : -1;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nseq, kvh, npart), dim3(256), 0, stream, out, part_acc, part_ml,
                       q, kc, vc, bt, sl, scale * kLog2e, nheads, kvh, nheads / kvh, block_size,
                       shift, max_blocks, alone);
  };
  if (npart > 1 && alone > 0) go(paged_decode_stream_kernel<HD, CT, true, true>);
  else if (npart > 1) go(paged_decode_stream_kernel<HD, CT, true, false>);
  else if (alone > 0) go(paged_decode_stream_kernel<HD, CT, false, true>);
  else go(paged_decode_stream_kernel<HD, CT, false, false>);
  if (npart > 1)
    hipLaunchKernelGGL((decode_stream_merge_kernel<HD>), dim3(nseq, nheads), dim3(HD), 0, stream,
                       out, part_acc, part_ml, sl, nheads, npart);
}

}  // namespace

int decode_alone_tiles(int nseq, int kvh, int group, int head_dim, bool fp8) {
  return alone_tiles(nseq, kvh, group, head_dim, fp8);
}

// Workgroups a sequence and key head may be cut over: enough for some six per CU
// where the batch alone has fewer (twice as many measured the same), at least four
// tiles each at the longest context.
int decode_stream_num_partitions(int nseq, int kvh, int max_context) {
  const int heads = nseq * kvh > 0 ? nseq * kvh : 1;
  const int tiles = (max_context + kTile - 1) / kTile;
  const int most = tiles / kMinTiles > 0 ? tiles / kMinTiles : 1;
  int npart = (1536 + heads - 1) / heads;
  if (npart > 64) npart = 64;
  return npart < most ? npart : most;
}

template <typename CT>
static void launch_hd(__hip_bfloat16* out, float* part_acc, float* part_ml,
                      const __hip_bfloat16* q, const CT* kc, const CT* vc, const int* bt,
                      const int* sl, float scale, int nseq, int nheads, int kvh, int head_dim,
                      int block_size, int max_blocks, int npart, hipStream_t stream) {
  if (head_dim == 64)
    launch<64, CT>(out, part_acc, part_ml, q, kc, vc, bt, sl, scale, nseq, nheads, kvh,
                   block_size, max_blocks, npart, stream);
  else
    launch<128, CT>(out, part_acc, part_ml, q, kc, vc, bt, sl, scale, nseq, nheads, kvh,
                    block_size, max_blocks, npart, stream);
}

void launch_paged_decode_stream(__hip_bfloat16* out, float* part_acc, float* part_ml,
                                const __hip_bfloat16* q, const __hip_bfloat16* kc,
                                const __hip_bfloat16* vc, const int* bt, const int* sl,
                                float scale, int nseq, int nheads, int kvh, int head_dim,
                                int block_size, int max_blocks, int npart, hipStream_t stream) {
  launch_hd(out, part_acc, part_ml, q, kc, vc, bt, sl, scale, nseq, nheads, kvh, head_dim,
            block_size, max_blocks, npart, stream);
}

void launch_paged_decode_stream_fp8(__hip_bfloat16* out, float* part_acc, float* part_ml,
                                    const __hip_bfloat16* q, const unsigned char* kc,
                                    const unsigned char* vc, const int* bt, const int* sl,
                                    float scale, int nseq, int nheads, int kvh, int head_dim,
                                    int block_size, int max_blocks, int npart,
                                    hipStream_t stream) {
  launch_hd(out, part_acc, part_ml, q, kc, vc, bt, sl, scale, nseq, nheads, kvh, head_dim,
            block_size, max_blocks, npart, stream);
}
