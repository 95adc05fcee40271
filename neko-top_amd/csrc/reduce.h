// reduce.h -- deterministic reductions for gfx950 (64-wide wavefronts).
//
// Every sum is taken with a fixed tree: one over the 64 lanes, then
// the wavefront partials of a block in order, then (in a one-block finalise
// kernel) the block partials in a fixed strided order.  For a given problem
// size the result is the same bit pattern on every run.
#pragma once
#include <hip/hip_runtime.h>

namespace nekoamd {

// The wave's sum of v in every lane (all 64 active), by lane moves of the
// vector unit: within a row of 16 by quad permutes and mirrors, then row 0
// into 1 and 2 into 3, then 1 into 3.  A butterfly of shuffles goes through
// LDS twelve times; where a workgroup reduces a value per basis vector that
// was as much work as the pass itself (mdot.h).
template <int CTRL, int ROWS>
__device__ __forceinline__ double lane_moved(double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (uint32_t)b, CTRL, ROWS, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (uint32_t)(b >> 32), CTRL, ROWS, 0xf, false);
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
__device__ __forceinline__ double wave_sum(double v) {
  // rounded here: a product must not be contracted into the first addition
  // in one kernel and not in another
  asm volatile("" : "+v"(v));
  v += lane_moved<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
  v += lane_moved<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
  v += lane_moved<0x141, 0xf>(v);  // row_half_mirror
  v += lane_moved<0x140, 0xf>(v);  // row_mirror
  v += lane_moved<0x142, 0xa>(v);  // row_bcast15 into rows 1 and 3
  v += lane_moved<0x143, 0xc>(v);  // row_bcast31 into rows 2 and 3
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, 63);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), 63);
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}

// Sum over a block of BS threads (BS a multiple of 64).  sh: BS/64 doubles of
// LDS.  The result is valid on thread 0.
template <int BS>
__device__ __forceinline__ double block_sum(double v, double* sh) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) sh[wv] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < BS / 64; ++q) s += sh[q];
  }
  __syncthreads();
  return s;
}

// Sum of n partials by one block of BS threads; valid on thread 0.
template <int BS>
__device__ __forceinline__ double sum_partials(const double* __restrict__ p,
                                               int64_t n, double* sh) {
  double s = 0.0;
  for (int64_t q = threadIdx.x; q < n; q += BS) s += p[q];
  return block_sum<BS>(s, sh);
}

constexpr int kRedBlock = 256;   // threads per block of a reducing kernel
constexpr int kRedGrid = 2048;   // max blocks (= partials) of one reduction
constexpr int kFinBlock = 1024;  // threads of the finalise kernel

}  // namespace nekoamd
