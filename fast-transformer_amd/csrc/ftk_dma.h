// Direct-to-LDS loads and the explicit waits around them, shared by the kernels
// that keep a per-wave LDS ring (RING and the LDS-fed MFMA form).
#pragma once

#include "ftk_device.h"

namespace ftk {

typedef __attribute__((address_space(1))) const void global_void_t;
typedef __attribute__((address_space(3))) void lds_void_t;

// 16 bytes per lane from `src` into LDS at dst + 16 lane (dst is wave-uniform).
// AUX 2: non-temporal (the weights, read once per call); 0: cached (x).
template <int AUX>
__device__ __forceinline__ void dma16(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds((global_void_t*)src, (lds_void_t*)dst, 16, 0, AUX);
}

// Wait until at most N vector memory instructions of this wave are outstanding.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Workgroup barrier for LDS traffic only. __syncthreads() also waits for every
// vector memory operation (vmcnt(0)), which would empty the ring mid-walk.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Byte address of an LDS object, as the ds instructions take it.
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

}  // namespace ftk
