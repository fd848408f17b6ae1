// Device-wide sums finished within the launch that forms them: every block
// leaves its partials and the last one to arrive adds them, in a fixed order.
#pragma once

#include "common.hpp"

namespace tpic_mi {

// Sum over the wave, valid in lane 0.
__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// The last block of a launch to finish adds what the others left. Only
// `partials` values and the arrival counters (zero between launches) pass
// between blocks within a launch: both are agent-scope accesses, which go past
// the XCDs' caches, and a block waits for its stores of partials before it
// arrives. (An agent-scope release instead writes back the XCD's whole L2 for
// every block: 33 us instead of 20 for an orthogonalisation at 100,000 nodes.)
__device__ __forceinline__ void put_partial(double* at, double v) {
  __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get_partial(const double* at) {
  return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Counters of one launch's arrivals, in words: a root, then one per kGroup
// blocks, each on a cache line of its own. Arrivals at one address follow one
// another at about 20 ns (1024 blocks at one counter: 20 us), so a block
// arrives at its group's and the last of a group at the root.
constexpr unsigned kGroup = 32, kCounterStride = 32, kMaxBlocks = 2048;
constexpr unsigned kCounters = (1 + kMaxBlocks / kGroup) * kCounterStride;

__device__ __forceinline__ bool arrive(unsigned* counter, unsigned expected) {
  if (__hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != expected - 1) return false;
  __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// True in every thread of the last of `blocks` blocks to get here. Thread 0's
// wave must have stored the block's partials itself.
__device__ __forceinline__ bool last_to_arrive(unsigned* counters, unsigned block, unsigned blocks, bool* lds) {
  if (threadIdx.x == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned group = block / kGroup, begin = group * kGroup;
    const unsigned size = blocks - begin < kGroup ? blocks - begin : kGroup;
    *lds = arrive(counters + (1 + group) * kCounterStride, size) && arrive(counters, (blocks + kGroup - 1) / kGroup);
  }
  __syncthreads();
  return *lds;
}

}  // namespace tpic_mi
