// uniform.h -- operator matrices that are the same for every lane, read row
// by row through the scalar data path.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace nekoamd {

// p as a pointer into the constant address space, made opaque to the
// compiler by an empty asm that also takes `dep` (a value of the previous
// row's sums) and uniform by readfirstlane: loads through it are scalar
// loads (read-only memory, the same address in every lane) that cannot be
// issued before dep is computed, so one matrix row at a time is live in
// scalar registers.  p must be the same in every lane.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T*
uniform_row(const T* p, const T& dep) {
  uint64_t v = (uint64_t)p;
  asm volatile("" : "+s"(v) : "v"(dep));
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const __attribute__((address_space(4))) T*)(((uint64_t)hi << 32) |
                                                       lo);
}

}  // namespace nekoamd
