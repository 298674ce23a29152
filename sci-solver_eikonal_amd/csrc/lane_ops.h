// lane_ops.h -- operations of a lane or wave that are written as instructions (device code).
//
// They stand apart from the code that uses them so that the visits and their scheduler (resident.h,
// visit_loop.h, block_sched.h) can be built for the host with other definitions of these few
// (tests/cpp/simt).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace eik {

// Waits until this wave's memory operations have completed at the device's coherence point
// (vmcnt covers loads, stores and atomics, with or without a result).
__device__ __forceinline__ void wait_memory() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Two non-negative values as fp16, rounded towards zero.
__device__ __forceinline__ uint32_t half_pair(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
}

// Copies 16 bytes per lane from memory straight to LDS (lane i of the wave to base + 16 i), so that
// no register holds them on the way.
__device__ __forceinline__ void copy_to_lds(const uint4* from, uint4* wave_base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                   (__attribute__((address_space(3))) void*)wave_base, 16, 0, 0);
}

// Adds to an LDS counter, by one lane, without the scan over the lanes that the compiler makes of an
// atomic with a result; returns the value before.
__device__ __forceinline__ int lds_take(int* counter, int n) {
  int old;
  asm volatile("ds_add_rtn_u32 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)"
               : "=v"(old)
               : "v"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) int*)counter), "v"(n)
               : "memory");
  return old;
}

// LDS atomics without a result, of one lane, as they are (see lds_take).  The caller waits for them
// (wait_memory) before its barrier.
__device__ __forceinline__ void lds_min(unsigned* p, unsigned v) {
  asm volatile("ds_min_u32 %0, %1"
               :: "v"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned*)p), "v"(v)
               : "memory");
}
__device__ __forceinline__ void lds_or(unsigned* p, unsigned v) {
  asm volatile("ds_or_b32 %0, %1"
               :: "v"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned*)p), "v"(v)
               : "memory");
}

}  // namespace eik
