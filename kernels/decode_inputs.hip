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
  if (tid < 3) {
    long* to = tid == 0 ? ids : tid == 1 ? positions : slots;
    to[row] = fresh(packed + (long)tid * n + row);
  } else if (tid == 3) {
    lens[row] = fresh(ints + row);
  } else if (tid == 4 && states != nullptr) {
    states[row] = fresh(ints + n + row);
  }
  const int* table = ints + 2L * n + (long)row * w;
  for (int j = tid; j < max_blocks; j += 256)
    tables[(long)row * max_blocks + j] = j < w ? fresh(table + j) : 0;
}

}  // namespace

void launch_decode_inputs(const long* packed, long* ids, long* positions, long* slots, int* lens,
                          int* states, int* tables, int n, int w, int rows, int max_blocks,
                          hipStream_t stream) {
  hipLaunchKernelGGL(decode_inputs_kernel, dim3(rows), dim3(256), 0, stream, packed, ids, positions,
                     slots, lens, states, tables, n, w, max_blocks);
}
