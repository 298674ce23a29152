// The operations of csrc/lane_ops.h for the host model (hip/hip_runtime.h beside this file).
#pragma once

#include <hip/hip_runtime.h>

namespace eik {

inline void wait_memory() { simt::wait(); }

// fp16 towards zero, of values that are not negative
inline uint32_t half_down(float x) {
  _Float16 h = (_Float16)x;
  if ((float)h > x) {
    uint16_t u;
    __builtin_memcpy(&u, &h, 2);
    --u;
    return u;
  }
  uint16_t u;
  __builtin_memcpy(&u, &h, 2);
  return u;
}
inline uint32_t half_pair(float a, float b) { return half_down(a) | half_down(b) << 16; }
inline void copy_to_lds(const uint4* from, uint4* wave_base) { wave_base[simt::me().lane] = *from; }
inline int lds_take(int* counter, int n) { return atomicAdd(counter, n); }
inline void lds_min(unsigned* p, unsigned v) { atomicMin(p, v); }
inline void lds_or(unsigned* p, unsigned v) { atomicOr(p, v); }

}  // namespace eik
