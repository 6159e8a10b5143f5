// A decode step's inputs from one packed buffer of pinned host memory into the static buffers
// of its captured graph:
//   int64 ids [n], positions [n], cache slots [n]; int32 lengths [n], state slots [n],
//   block tables [n, w]
// Rows from n to the graph's `rows` get slot -1, length 0 and state slot -1, tables zeros past
// w.  One launch that reads over the bus for what were ten copies and up to four fills, 3 us
// each: a step of one stream 363 -> 344 us (llama-1b), 451 -> 434 (llama-3-8b, 4 bits).
//
// The buffer is written again two steps later, at the same address: system-scope loads, which
// no cache answers.

#include "common.h"

namespace {

template <typename T> DEVINLINE T fresh(const T* at) {
  return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// grid (rows)
__global__ __launch_bounds__(256) void decode_inputs_kernel(
    const long* __restrict__ packed, long* __restrict__ ids, long* __restrict__ positions,
    long* __restrict__ slots, int* __restrict__ lens, int* __restrict__ states,   // or null
    int* __restrict__ tables, const int n, const int w, const int max_blocks) {
  const int row = blockIdx.x, tid = threadIdx.x;
  const int* ints = reinterpret_cast<const int*>(packed + 3L * n);
  if (row >= n) {
    if (tid == 0) {
      slots[row] = -1;
      lens[row] = 0;
      if (states != nullptr) states[row] = -1;
    }
    return;
  }
  // one trip over the bus: the first wave has the row's numbers, a word a thread, the others
  // its table (in branches one after the other, each with its load and store: one row of 15 blocks
  // 5.5 us, now 3.0; of 500 6.5, 3.0; 16 of 300 10.8, 6.0; 300 of 32 8.9, 7.7)
  if (tid < 64) {
    const int* word = nullptr;
    int* to = nullptr;
    if (tid < 6) {
      word = reinterpret_cast<const int*>(packed + (long)(tid / 2) * n + row) + tid % 2;
      to = reinterpret_cast<int*>((tid < 2 ? ids : tid < 4 ? positions : slots) + row) + tid % 2;
    } else if (tid == 6) {
      word = ints + row;
      to = lens + row;
    } else if (tid == 7 && states != nullptr) {
      word = ints + n + row;
      to = states + row;
    }
    if (word != nullptr) *to = fresh(word);
    return;
  }
  const int* table = ints + 2L * n + (long)row * w;
  int* out = tables + (long)row * max_blocks;
  constexpr int AHEAD = 4, STRIDE = 192;
  for (int j0 = tid - 64; j0 < max_blocks; j0 += AHEAD * STRIDE) {
    int v[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      v[i] = 0;
      if (j0 + i * STRIDE < w) v[i] = fresh(table + j0 + i * STRIDE);
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (j0 + i * STRIDE < max_blocks) out[j0 + i * STRIDE] = v[i];
  }
}

}  // namespace

void launch_decode_inputs(const long* packed, long* ids, long* positions, long* slots, int* lens,
                          int* states, int* tables, int n, int w, int rows, int max_blocks,
                          hipStream_t stream) {
  hipLaunchKernelGGL(decode_inputs_kernel, dim3(rows), dim3(256), 0, stream, packed, ids, positions,
                     slots, lens, states, tables, n, w, max_blocks);
}
