// SiLU-mul activation, NeoX rotary embedding, paged-KV cache write
// support.  All memory-bound: 16-B vector accesses, f32 math.

#include "common.h"

// ---------------------------------------------------------------------------
// silu_and_mul: out[t, i] = silu(x[t, i]) * x[t, d + i]
// ---------------------------------------------------------------------------

// grid (rows, pieces of a row): a vector a thread, so that a few rows are not a chain of
// loads (61 rows of 14336: 5.4 -> 4.1 us)
template <typename T>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(
    T* __restrict__ out,        // [rows, d]
    const T* __restrict__ x,    // [rows, 2*d]
    const int d) {
  constexpr int V = Vec16<T>::kElems;
  const int row = blockIdx.x, i = (blockIdx.y * 256 + threadIdx.x) * V;
  if (i >= d) return;
  const T* a_row = x + (long)row * 2 * d;
  Vec16<T> a = load16(a_row + i);
  Vec16<T> b = load16(a_row + d + i);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    float av = ScalarOps<T>::to_f32(a.data[j]);
    float bv = ScalarOps<T>::to_f32(b.data[j]);
    float s = av / (1.f + __expf(-av));
    a.data[j] = ScalarOps<T>::from_f32(s * bv);
  }
  store16(out + (long)row * d + i, a);
}

template <typename T>
void launch_silu_and_mul(T* out, const T* x, int rows, int d, hipStream_t s) {
  constexpr int kPiece = 256 * Vec16<T>::kElems;
  hipLaunchKernelGGL(silu_and_mul_kernel<T>, dim3(rows, (d + kPiece - 1) / kPiece), dim3(256), 0,
                     s, out, x, d);
}

// ---------------------------------------------------------------------------
// NeoX rotary embedding: q into q_out (dense rows, may be q itself), k in place.
// Rows of q and k may lie further apart than they are long (column slices of one
// projection).
// cos_sin_cache: [max_pos, head_dim] f32, first half cos, second half sin.
// One block per token; threads cover (head, i<half) pairs for q then k.
// ---------------------------------------------------------------------------

template <typename T>
__global__ void rotary_embedding_kernel(
    const long* __restrict__ positions,  // [T]
    T* q_out,                            // [T, nq * hd]
    const T* q,                          // [T, nq * hd], rows q_stride apart
    T* __restrict__ k,                   // [T, nk * hd], rows k_stride apart
    const float* __restrict__ cos_sin,   // [max_pos, hd]
    const int nq, const int nk, const int hd, const long q_stride, const long k_stride) {
  const int token = blockIdx.x;
  const long pos = positions[token];
  const float* cs = cos_sin + pos * hd;
  const int half = hd / 2;

  const T* q_row = q + token * q_stride;
  T* o_row = q_out + (long)token * nq * hd;
  T* k_row = k + token * k_stride;
  const int total = (nq + nk) * half;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int h = idx / half;
    const int i = idx % half;
    const T* row = h < nq ? q_row + h * hd : k_row + (h - nq) * hd;
    T* out = h < nq ? o_row + h * hd : k_row + (h - nq) * hd;
    const float c = cs[i];
    const float s = cs[half + i];
    const float x1 = ScalarOps<T>::to_f32(row[i]);
    const float x2 = ScalarOps<T>::to_f32(row[i + half]);
    out[i] = ScalarOps<T>::from_f32(x1 * c - x2 * s);
    out[i + half] = ScalarOps<T>::from_f32(x2 * c + x1 * s);
  }
}

template <typename T>
void launch_rotary_embedding(const long* positions, T* q_out, const T* q, T* k,
                             const float* cos_sin, int tokens, int nq, int nk,
                             int hd, long q_stride, long k_stride, hipStream_t s) {
  int threads = 256;
  hipLaunchKernelGGL(rotary_embedding_kernel<T>, dim3(tokens), dim3(threads), 0,
                     s, positions, q_out, q, k, cos_sin, nq, nk, hd, q_stride, k_stride);
}

// ---------------------------------------------------------------------------
// reshape_and_cache: scatter per-token K/V rows into the paged cache.
// cache layout: [num_blocks, block_size, kv_heads, head_dim] — a token's
// (kv_heads*head_dim) row is contiguous, so this is a straight 16-B copy.  Rows
// of k and v may lie k_stride / v_stride elements apart.
// ---------------------------------------------------------------------------

template <typename T>
__global__ void reshape_and_cache_kernel(
    const T* __restrict__ k,      // [T, kvh * hd]
    const T* __restrict__ v,
    T* __restrict__ k_cache,      // [nb * bs, kvh * hd] flattened
    T* __restrict__ v_cache,
    const long* __restrict__ slots,  // [T]
    const int row_elems, const long k_stride, const long v_stride) {
  constexpr int V = Vec16<T>::kElems;
  const int token = blockIdx.x;
  const long slot = slots[token];
  if (slot < 0) return;
  const T* k_src = k + token * k_stride;
  const T* v_src = v + token * v_stride;
  T* k_dst = k_cache + slot * row_elems;
  T* v_dst = v_cache + slot * row_elems;
  for (int i = threadIdx.x * V; i < row_elems; i += blockDim.x * V) {
    store16(k_dst + i, load16(k_src + i));
    store16(v_dst + i, load16(v_src + i));
  }
}

template <typename T>
void launch_reshape_and_cache(const T* k, const T* v, T* kc, T* vc,
                              const long* slots, int tokens, int row_elems,
                              long k_stride, long v_stride, hipStream_t s) {
  int threads = 128;
  hipLaunchKernelGGL(reshape_and_cache_kernel<T>, dim3(tokens), dim3(threads),
                     0, s, k, v, kc, vc, slots, row_elems, k_stride, v_stride);
}

// fp8 KV cache: bf16 K/V quantized to OCP e4m3
// at cache-write time; halves the decode-attention HBM stream and doubles
// KV capacity in the 288 GB pool.
__global__ void reshape_and_cache_fp8_kernel(
    const __hip_bfloat16* __restrict__ k,  // [T, kvh * hd]
    const __hip_bfloat16* __restrict__ v,
    unsigned char* __restrict__ k_cache,   // [nb * bs, kvh * hd] e4m3
    unsigned char* __restrict__ v_cache,
    const long* __restrict__ slots,
    const int row_elems, const long k_stride, const long v_stride) {
  const int token = blockIdx.x;
  const long slot = slots[token];
  if (slot < 0) return;
  const __hip_bfloat16* k_src = k + token * k_stride;
  const __hip_bfloat16* v_src = v + token * v_stride;
  unsigned char* k_dst = k_cache + slot * row_elems;
  unsigned char* v_dst = v_cache + slot * row_elems;
  for (int i = threadIdx.x * 8; i < row_elems; i += blockDim.x * 8) {
    *reinterpret_cast<u32x2_vec_t*>(k_dst + i) = bf16x8_to_fp8x8(
        *reinterpret_cast<const bf16x8_vec_t*>(k_src + i));
    *reinterpret_cast<u32x2_vec_t*>(v_dst + i) = bf16x8_to_fp8x8(
        *reinterpret_cast<const bf16x8_vec_t*>(v_src + i));
  }
}

void launch_reshape_and_cache_fp8(const __hip_bfloat16* k,
                                  const __hip_bfloat16* v, unsigned char* kc,
                                  unsigned char* vc, const long* slots,
                                  int tokens, int row_elems, long k_stride,
                                  long v_stride, hipStream_t s) {
  hipLaunchKernelGGL(reshape_and_cache_fp8_kernel, dim3(tokens), dim3(128), 0,
                     s, k, v, kc, vc, slots, row_elems, k_stride, v_stride);
}

// ---------------------------------------------------------------------------
// Both at once, for bf16: q turned into dense rows, k turned on its way into the cache
// (rounded to bf16 first, as if it had been kept), v copied.  Eight neighbours of each
// half of a head a thread, a workgroup 256 of a token's pieces.
//
// Bound by latency at decode sizes, where rotation and cache write apart were 5.0 + 4.3 us
// (one row of 32/8 heads of 128, traced): a step of one stream, 8 layers, llama-1b 434 ->
// 413 us, llama-3-8b in 4 bits 638 -> 602.
// ---------------------------------------------------------------------------
template <bool FP8>
__global__ __launch_bounds__(256) void rotary_cache_kernel(
    const long* __restrict__ positions, __hip_bfloat16* q_out, const __hip_bfloat16* q,
    const __hip_bfloat16* __restrict__ k, const __hip_bfloat16* __restrict__ v,
    const float* __restrict__ cos_sin, unsigned char* __restrict__ k_cache,
    unsigned char* __restrict__ v_cache, const long* __restrict__ slots, const int nq,
    const int nk, const int hd, const long q_stride, const long k_stride, const long v_stride,
    const int blocks) {
  const long token = blockIdx.x / blocks;
  const int piece = blockIdx.x % blocks * 256 + threadIdx.x;
  const int half = hd / 2, per = half / 8, turned = (nq + nk) * per;
  const long slot = slots[token];
  auto cache = [&](unsigned char* to, long at, const bf16x8_vec_t& x) {
    if constexpr (FP8)
      *reinterpret_cast<u32x2_vec_t*>(to + at) = bf16x8_to_fp8x8(x);
    else
      *reinterpret_cast<bf16x8_vec_t*>(to + at * 2) = x;
  };
  const long row = slot * nk * hd;
  if (piece < turned) {
    const int h = piece / per, i = piece % per * 8;
    const bool key = h >= nq;
    if (key && slot < 0) return;
    const __hip_bfloat16* from =
        key ? k + token * k_stride + (h - nq) * hd : q + token * q_stride + h * hd;
    const Vec16<__hip_bfloat16> a = load16(from + i), b = load16(from + half + i);
    const float* cs = cos_sin + positions[token] * hd + i;
    union { __hip_bfloat16 e[8]; bf16x8_vec_t v; } lo, hi;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float c = cs[j], s = cs[half + j];
      const float x1 = __bfloat162float(a.data[j]), x2 = __bfloat162float(b.data[j]);
      lo.e[j] = __float2bfloat16(x1 * c - x2 * s);
      hi.e[j] = __float2bfloat16(x2 * c + x1 * s);
    }
    if (key) {
      const long at = row + (h - nq) * hd + i;
      cache(k_cache, at, lo.v);
      cache(k_cache, at + half, hi.v);
    } else {
      __hip_bfloat16* to = q_out + (token * nq + h) * hd + i;
      *reinterpret_cast<bf16x8_vec_t*>(to) = lo.v;
      *reinterpret_cast<bf16x8_vec_t*>(to + half) = hi.v;
    }
  } else if (piece - turned < nk * hd / 8 && slot >= 0) {
    const int i = (piece - turned) * 8;
    cache(v_cache, row + i, *reinterpret_cast<const bf16x8_vec_t*>(v + token * v_stride + i));
  }
}

// hd % 16 == 0, rows of q, k and v 16-byte aligned
void launch_rotary_cache(const long* positions, __hip_bfloat16* q_out, const __hip_bfloat16* q,
                         const __hip_bfloat16* k, const __hip_bfloat16* v, const float* cos_sin,
                         void* k_cache, void* v_cache, const long* slots, int tokens, int nq,
                         int nk, int hd, long q_stride, long k_stride, long v_stride, bool fp8,
                         hipStream_t s) {
  const int pieces = (nq + nk) * (hd / 16) + nk * hd / 8, blocks = (pieces + 255) / 256;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)tokens * blocks), dim3(256), 0, s, positions, q_out,
                       q, k, v, cos_sin, static_cast<unsigned char*>(k_cache),
                       static_cast<unsigned char*>(v_cache), slots, nq, nk, hd, q_stride,
                       k_stride, v_stride, blocks);
  };
  if (fp8) go(rotary_cache_kernel<true>);
  else go(rotary_cache_kernel<false>);
}

#define INSTANTIATE(T)                                                         \
  template void launch_silu_and_mul<T>(T*, const T*, int, int, hipStream_t);   \
  template void launch_rotary_embedding<T>(const long*, T*, const T*, T*,      \
                                           const float*, int, int, int, int,   \
                                           long, long, hipStream_t);           \
  template void launch_reshape_and_cache<T>(const T*, const T*, T*, T*,        \
                                            const long*, int, int, long, long, \
                                            hipStream_t);

INSTANTIATE(float)
INSTANTIATE(__hip_bfloat16)
INSTANTIATE(__half)
