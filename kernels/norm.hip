// Fused RMSNorm kernels.
// Memory-bound: one workgroup per row, 16-B vector loads (scalar
// bf16 loads cost ~2x), sum-of-squares in f32, one pass read + one pass write.
//
// Of a step's rows what counts is the chain of latencies.  Rows of up to 8192 (f32: 4096)
// stay in registers, a vector a thread (many rows without a sum: two or four), the weight is asked
// for with the row, and the waves' sums meet once, which no store is waited for at: us at 256
// threads, the sum stored first | here: 1 row of 4096 2.4 | 2.0, 61 3.3 | 2.8, 1000 9.9 | 9.1, 8192
// 50.7 | 49.1; 64 of 8192 4.6 | 3.4.
// (Rows read again after the sum, which waited for a cold weight: 61 of 4096 4.3 where 3.7.)

#include "common.h"

namespace {

// the workgroup's sum, in one meeting of its WAVES
template <int WAVES>
DEVINLINE float sum_of_waves(float x, float* lds) {
  x = wave_reduce_sum(x);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = x;
  __syncthreads();
  float sum = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; w += 4) sum += (lds[w] + lds[w + 1]) + (lds[w + 2] + lds[w + 3]);
  return sum;
}

// x <- rmsnorm(x + residual) w, residual <- x + residual, or (ADD false) out <- rmsnorm(x) w;
// hidden is a multiple of a vector and at most CHUNKS of them a thread
template <typename T, int THREADS, int CHUNKS, bool ADD>
__global__ __launch_bounds__(THREADS) void rms_norm_row_kernel(
    T* out, const T* x, T* residual, const T* __restrict__ weight, const float eps,
    const int hidden) {
  constexpr int V = Vec16<T>::kElems;
  const long row = (long)blockIdx.x * hidden;
  Vec16<T> v[CHUNKS], r[CHUNKS], w[CHUNKS];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = (c * THREADS + threadIdx.x) * V;
    if (i >= hidden) continue;
    v[c] = load16(x + row + i);
    if (ADD) r[c] = load16(residual + row + i);
    w[c] = load16(weight + i);
  }
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = (c * THREADS + threadIdx.x) * V;
    if (i >= hidden) continue;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      // the norm is of the rounded sum, which is what is stored
      if (ADD)
        v[c].data[j] = ScalarOps<T>::from_f32(ScalarOps<T>::to_f32(v[c].data[j]) +
                                              ScalarOps<T>::to_f32(r[c].data[j]));
      const float s = ScalarOps<T>::to_f32(v[c].data[j]);
      ss += s * s;
    }
  }
  __shared__ float lds[THREADS / 64];
  const float inv = rsqrtf(sum_of_waves<THREADS / 64>(ss, lds) / hidden + eps);
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = (c * THREADS + threadIdx.x) * V;
    if (i >= hidden) continue;
    if (ADD) store16(residual + row + i, v[c]);   // (the meeting would wait for it)
#pragma unroll
    for (int j = 0; j < V; ++j)
      v[c].data[j] = ScalarOps<T>::from_f32(ScalarOps<T>::to_f32(v[c].data[j]) * inv *
                                            ScalarOps<T>::to_f32(w[c].data[j]));
    store16(out + row + i, v[c]);
  }
}

template <typename T, bool ADD>
bool launch_row(T* out, const T* x, T* residual, const T* w, float eps, int rows, int hidden,
                hipStream_t stream) {
  constexpr int V = Vec16<T>::kElems;
  if (hidden % V != 0) return false;
  auto go = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(threads), 0, stream, out, x, residual, w, eps,
                       hidden);
    return true;
  };
  if (hidden <= 256 * V) return go(rms_norm_row_kernel<T, 256, 1, ADD>, 256);
  if constexpr (!ADD) {
    // Many rows are bytes, of which a wave with two vectors or four has more on their way.  us, a vector a
    // thread | 256 threads: 512 x 4096 3.7 | 3.8, 512 x 6144 4.5 | 4.5, 1000 x 5120 6.4 | 5.7, 1500 x
    // 4096 6.9 | 6.2, 1500 x 6144 10.3 | 8.0, 8192 x 4096 24.7 | 23.9, 8192 x 5120 37.7 | 30.5; with the sum,
    // twice the bytes, 1000 x 4096 9.2 | 9.5, 8192 x 4096 48.6 | 51.2.
    if (rows > 768 && hidden <= 512 * V) return go(rms_norm_row_kernel<T, 256, 2, ADD>, 256);
    if (rows > 768 && hidden <= 1024 * V) return go(rms_norm_row_kernel<T, 256, 4, ADD>, 256);
  }
  if (hidden <= 512 * V) return go(rms_norm_row_kernel<T, 512, 1, ADD>, 512);
  if (hidden <= 1024 * V) return go(rms_norm_row_kernel<T, 1024, 1, ADD>, 1024);
  return false;
}

}  // namespace

template <typename T>
__global__ void rms_norm_kernel(
    T* __restrict__ out,          // [rows, hidden]
    const T* __restrict__ input,  // [rows, hidden]
    const T* __restrict__ weight, // [hidden]
    const float eps,
    const int hidden) {
  constexpr int V = Vec16<T>::kElems;
  const int row = blockIdx.x;
  const T* in_row = input + (long)row * hidden;
  T* out_row = out + (long)row * hidden;

  float ss = 0.f;
  for (int i = threadIdx.x * V; i < hidden; i += blockDim.x * V) {
    Vec16<T> v = load16(in_row + i);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      float x = ScalarOps<T>::to_f32(v.data[j]);
      ss += x * x;
    }
  }
  __shared__ float lds[16];
  ss = block_reduce_sum(ss, lds);
  const float inv = rsqrtf(ss / hidden + eps);

  for (int i = threadIdx.x * V; i < hidden; i += blockDim.x * V) {
    Vec16<T> v = load16(in_row + i);
    Vec16<T> w = load16(weight + i);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      float x = ScalarOps<T>::to_f32(v.data[j]) * inv *
                ScalarOps<T>::to_f32(w.data[j]);
      v.data[j] = ScalarOps<T>::from_f32(x);
    }
    store16(out_row + i, v);
  }
}

// x <- rmsnorm(x + residual) * w ; residual <- x + residual   (both in place)
template <typename T>
__global__ void fused_add_rms_norm_kernel(
    T* __restrict__ x,          // [rows, hidden]
    T* __restrict__ residual,   // [rows, hidden]
    const T* __restrict__ weight,
    const float eps,
    const int hidden) {
  constexpr int V = Vec16<T>::kElems;
  const int row = blockIdx.x;
  T* x_row = x + (long)row * hidden;
  T* r_row = residual + (long)row * hidden;

  float ss = 0.f;
  for (int i = threadIdx.x * V; i < hidden; i += blockDim.x * V) {
    Vec16<T> xv = load16(x_row + i);
    Vec16<T> rv = load16(r_row + i);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      float s = ScalarOps<T>::to_f32(xv.data[j]) + ScalarOps<T>::to_f32(rv.data[j]);
      rv.data[j] = ScalarOps<T>::from_f32(s);
      // re-read the rounded sum so the norm matches what is stored
      float sr = ScalarOps<T>::to_f32(rv.data[j]);
      ss += sr * sr;
    }
    store16(r_row + i, rv);
  }
  __shared__ float lds[16];
  ss = block_reduce_sum(ss, lds);
  const float inv = rsqrtf(ss / hidden + eps);

  for (int i = threadIdx.x * V; i < hidden; i += blockDim.x * V) {
    Vec16<T> rv = load16(r_row + i);
    Vec16<T> wv = load16(weight + i);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      float v = ScalarOps<T>::to_f32(rv.data[j]) * inv *
                ScalarOps<T>::to_f32(wv.data[j]);
      rv.data[j] = ScalarOps<T>::from_f32(v);
    }
    store16(x_row + i, rv);
  }
}

template <typename T>
void launch_rms_norm(T* out, const T* in, const T* w, float eps, int rows,
                     int hidden, hipStream_t stream) {
  if (launch_row<T, false>(out, in, nullptr, w, eps, rows, hidden, stream)) return;
  const int threads = 256;
  hipLaunchKernelGGL(rms_norm_kernel<T>, dim3(rows), dim3(threads), 0, stream,
                     out, in, w, eps, hidden);
}

template <typename T>
void launch_fused_add_rms_norm(T* x, T* res, const T* w, float eps, int rows,
                               int hidden, hipStream_t stream) {
  if (launch_row<T, true>(x, x, res, w, eps, rows, hidden, stream)) return;
  const int threads = 256;
  hipLaunchKernelGGL(fused_add_rms_norm_kernel<T>, dim3(rows), dim3(threads), 0,
                     stream, x, res, w, eps, hidden);
}

#define INSTANTIATE(T)                                                        \
  template void launch_rms_norm<T>(T*, const T*, const T*, float, int, int,   \
                                   hipStream_t);                              \
  template void launch_fused_add_rms_norm<T>(T*, T*, const T*, float, int,    \
                                             int, hipStream_t);

INSTANTIATE(float)
INSTANTIATE(__hip_bfloat16)
INSTANTIATE(__half)
