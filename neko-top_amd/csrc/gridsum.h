// gridsum.h -- sums over all workgroups of a running kernel, for solvers
// whose iterations are too short to be launches of their own.
//
// Every workgroup publishes its partial sums in a slot of its own and reads
// all slots: a reduction and a grid barrier in one exchange, without an
// atomic that the workgroups contend for.  A double travels as two 64-bit
// words of 32 value bits and a 32-bit tag, each stored and loaded whole at
// device scope, so a reader knows from the word itself whether it belongs to
// this exchange; tags must not repeat while an older word can still be in a
// slot (one counter per set of slots, advanced over launches).
//
// Other values cross the grid the same way (grid_put, grid_get): the reader
// waits for the very words it needs, so nothing has to be ordered before a
// publish.  A word may be overwritten once a later exchange has shown that
// every workgroup is past reading it.
//
// All workgroups must be resident at once: the launcher bounds the grid by
// the occupancy of an empty device.  A wait lasts at most `wait` ticks of the
// 100 MHz clock; a workgroup that gives up leaves, and so the others do.  To
// have the first wait given up at once, the launcher passes wait 0 and has
// the sums take one slot more than there are workgroups, which nobody fills
// (a test of the wait in the loop that polls costs 4 % of a small solve).
#pragma once
#include <hip/hip_runtime.h>

#include "reduce.h"

namespace nekoamd {

constexpr unsigned long long kGridTicks = 100;  // of the clock, per us
constexpr unsigned long long kGridWait = 1000000 * kGridTicks;  // default, 1 s

template <typename T>
__device__ __forceinline__ T dev_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void dev_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The calling thread's earlier dev_stores have reached the device's memory.
__device__ __forceinline__ void dev_stores_done() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

__device__ __forceinline__ void grid_put(uint64_t* s, uint32_t tag, double v) {
  const uint64_t hi = (uint64_t)tag << 32;
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  dev_store(s, (uint64_t)(hi | (b & 0xFFFFFFFFull)));
  dev_store(s + 1, (uint64_t)(hi | (b >> 32)));
}
// The N values at s[j], waited for together (their loads in flight at once);
// the first n of them count.  *fail = 1 if the wait was given up.
template <int N>
__device__ __forceinline__ void grid_get(const uint64_t* const (&s)[N], int n,
                                         uint32_t tag, unsigned long long wait,
                                         int* fail, double (&out)[N]) {
  const unsigned long long t0 = wall_clock64();
  for (;;) {
    uint64_t w[2 * N];
    bool here = true;
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (j < n) {
        w[2 * j] = dev_load(s[j]);
        w[2 * j + 1] = dev_load(s[j] + 1);
      }
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (j < n) {
        here &= (uint32_t)(w[2 * j] >> 32) == tag &&
                (uint32_t)(w[2 * j + 1] >> 32) == tag;
        out[j] = __longlong_as_double(
            (long long)((w[2 * j] & 0xFFFFFFFFull) | (w[2 * j + 1] << 32)));
      }
    if (here) return;
    if (wall_clock64() - t0 >= wait) {
      *fail = 1;
      return;
    }
  }
}

// One thread of a workgroup: its NV partial sums into slots[wg].
template <int NV>
__device__ __forceinline__ void grid_publish(uint64_t* slots, int wg,
                                             uint32_t tag,
                                             const double (&v)[NV]) {
#pragma unroll
  for (int j = 0; j < NV; ++j)
    grid_put(slots + ((int64_t)wg * NV + j) * 2, tag, v[j]);
}

// Every thread of a workgroup: the sums over the nwg slots of this tag, the
// same value in every thread of every workgroup (blockDim.x, a multiple of
// 64, must be the same in all).  Slots t, t + NT, .. are added by thread t <
// NT (0: blockDim.x), then as block_sum (reduce.h) adds.  sh: NV doubles per
// wave of the workgroup; *fail: a shared int that is 0, set if a wait was given up.  Returns false
// (in every thread) in that case.  sh may be written again after the next
// workgroup barrier.
template <int NV, int NT = 0>
__device__ __forceinline__ bool grid_sum(const uint64_t* slots, int nwg,
                                         uint32_t tag, unsigned long long wait,
                                         double* sh, int* fail,
                                         double (&out)[NV]) {
  double v[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) v[j] = 0.0;
  const int step = NT ? NT : (int)blockDim.x;
  for (int q = NT && (int)threadIdx.x >= NT ? nwg : (int)threadIdx.x; q < nwg;
       q += step) {
    const uint64_t* s[NV];
    double p[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) s[j] = slots + ((int64_t)q * NV + j) * 2;
    grid_get<NV>(s, NV, tag, wait, fail, p);
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] += p[j];
  }
  const int wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    v[j] = wave_sum(v[j]);
    if ((threadIdx.x & 63) == 0) sh[wv * NV + j] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NV; ++j) out[j] = 0.0;
  for (int k = 0; k < nw; ++k)
#pragma unroll
    for (int j = 0; j < NV; ++j) out[j] += sh[k * NV + j];
  return *fail == 0;
}

}  // namespace nekoamd
