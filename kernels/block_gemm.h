// What the tiled products share: loads from HBM straight to LDS (buffer_load ... lds, 16 bytes
// a lane), waits that leave later ones on their way, and the meeting of the waves.
#pragma once

#include "common.h"

namespace block_gemm {

typedef __attribute__((ext_vector_type(8))) short bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

template <int N> DEVINLINE void wait_loads() {
  static_assert(N < 64, "vmcnt has six bits");
  // vmcnt(N), other counters left alone
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}

// vmcnt(N) and lgkmcnt(0)
template <int N> DEVINLINE void wait_loads_and_reads() {
  static_assert(N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0070);
}

// The waves meet; loads on their way to LDS stay on their way (a fence would wait for
// all of them).
DEVINLINE void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// 4 GB (or less) from a wave-uniform address on
DEVINLINE __amdgpu_buffer_rsrc_t resource(const void* from, unsigned size = 0xffffffff) {
  const unsigned long long at = reinterpret_cast<unsigned long long>(from);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)at);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(at >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void*>((unsigned long long)hi << 32 | lo), 0, size, 0x00027000);
}

// 16 (4) bytes a lane from `from` + offset (+ the uniform ahead) to lds + 16 (4) lane.
// Buffer loads: with a global one on its way the compiler has every read of LDS wait for
// all reads before it.
template <int HINT = 0>
DEVINLINE void load_lds(char* lds, __amdgpu_buffer_rsrc_t from, unsigned offset, int ahead) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      from, (__attribute__((address_space(3))) void*)lds, 16, offset, ahead, 0, HINT);
}
DEVINLINE void load_lds4(char* lds, __amdgpu_buffer_rsrc_t from, unsigned offset, int ahead) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      from, (__attribute__((address_space(3))) void*)lds, 4, offset, ahead, 0, 0);
}

}  // namespace block_gemm
