// Global -> LDS streaming and hand-waited LDS fragment reads, shared by the tile pipelines (gfx950).
#pragma once
#include <utility>

#include "common.h"

namespace tread {

// 16 bytes per lane from global memory straight into LDS: lane l's bytes land at lds + 16 l
// (lds is wave-uniform).
__device__ __forceinline__ void lds_load16(const bf16_t* g, bf16_t* lds) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)(uintptr_t)lds, 16, 0, 0);
}

// The same for bytes that one work group reads once (aux 2: non-temporal): streamed weights.
__device__ __forceinline__ void lds_load16_nt(const bf16_t* g, bf16_t* lds) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)(uintptr_t)lds, 16, 0, 2);
}

// LDS byte address of a pointer into the work group's shared memory (the low 32 bits of its
// generic address; the LDS aperture is 4 GiB-aligned).
__device__ __forceinline__ uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)p; }

template <int OFF>
__device__ __forceinline__ bf16x8_t lds_read128(uint32_t addr) {
  u32x4_t r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
  return __builtin_bit_cast(bf16x8_t, r);
}
template <int N>
__device__ __forceinline__ void lgkm_wait(bf16x8_t& v) {
  asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v) : "n"(N));
}

template <int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Work-group barrier of the tile pipelines, after each wave has waited (vm_wait) for its own
// global->LDS loads of the tiles the barrier publishes. __syncthreads() would also wait for every
// outstanding vector memory operation (vmcnt(0)), i.e. for the tiles still being prefetched,
// taking the pipeline's load lead away at every barrier.
__device__ __forceinline__ void tile_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace tread
