// sc_block.h -- device helpers of whole blocks: sums over a block, and the door
// and barriers of launches that run several dependent passes.
#ifndef SIMCORE_AMD_BLOCK_H_
#define SIMCORE_AMD_BLOCK_H_

#include <hip/hip_runtime.h>

#include "sc_internal.h"

namespace sc {

// Sum of v over each SUB consecutive threads of a block; `ws` holds one int
// per wavefront of the block.
template <int SUB>
__device__ __forceinline__ int block_sum(int v, int *ws) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
  __syncthreads();
  const int w0 = (int)threadIdx.x / SUB * (SUB / 64);
  int t = 0;
#pragma unroll
  for (int i = 0; i < SUB / 64; ++i) t += ws[w0 + i];
  __syncthreads();
  return t;
}

// exclusive scan of v over each SUB consecutive threads
template <int SUB>
__device__ __forceinline__ int block_excl(int v, int *total, int *ws) {
  const int lane = threadIdx.x & 63, w0 = (int)threadIdx.x / SUB * (SUB / 64);
  const int w = ((int)threadIdx.x >> 6) - w0;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) ws[threadIdx.x >> 6] = x;
  __syncthreads();
  int base = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < SUB / 64; ++i) {
    const int t = ws[w0 + i];
    if (i < w) base += t;
    tot += t;
  }
  __syncthreads();
  *total = tot;
  return base + x - v;
}

// Passes of one launch with barriers between them.  A barrier never waits for
// a block that is not running: the blocks that take part are those that have
// arrived when the first of them closes the door -- when all have, or after
// kDoorTicks -- and a block that arrives later leaves at once.  The passes
// take their block index and count from that, so any number of blocks (one,
// if need be) does all the work.  A barrier takes 3.5 us among 64 blocks, 7
// among 256, 12 among 512 (device-scope release and acquire included).
constexpr uint32_t kDoorClosed = 0x80000000u;
constexpr long long kDoorTicks = 2000;  // of the 100 MHz clock: 20 us

__device__ __forceinline__ uint32_t bar_load(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t bar_add(uint32_t *p) {
  return __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// All threads: enters the block; false when it came too late.  *rank and
// *parts: its number among the blocks taking part, and how many those are.
// `blocks`: those of the launch that belong to the system.
__device__ __forceinline__ bool door_enter(Door *b, uint32_t blocks, int *rank,
                                           int *parts) {
  __shared__ uint32_t sr, sp;
  if (threadIdx.x == 0) {
    const uint32_t r = bar_add(&b->arrived);
    uint32_t p = 0;
    if (r == 0) {  // the first to arrive closes the door
      const long long t0 = wall_clock64();
      while (bar_load(&b->arrived) < blocks && wall_clock64() - t0 < kDoorTicks)
        __builtin_amdgcn_s_sleep(1);
      p = __hip_atomic_fetch_or(&b->arrived, kDoorClosed, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&b->parts, p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else if (!(r & kDoorClosed)) {
      while ((p = bar_load(&b->parts)) == 0) __builtin_amdgcn_s_sleep(1);
    }
    sr = r;
    sp = p;
  }
  __syncthreads();
  *rank = (int)(sr & ~kDoorClosed);
  *parts = (int)sp;
  return !(sr & kDoorClosed);
}

// Barrier `k` of a launch among the `parts` blocks inside (all threads).  The
// arrivals are counted in kBarGroups groups and the full groups in one word,
// as atomics on one address serialise.
__device__ __forceinline__ void bar_wait(Door *b, int k, int rank, int parts) {
  __syncthreads();
  if (parts > 1 && threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const int grp = rank % kBarGroups;
    const uint32_t size = (uint32_t)((parts - grp + kBarGroups - 1) / kBarGroups);
    const uint32_t groups = (uint32_t)(parts < kBarGroups ? parts : kBarGroups);
    if (bar_add(&b->group[k][grp][0]) + 1 == size) bar_add(&b->full[k][0]);
    while (bar_load(&b->full[k][0]) < groups) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
}

// Every block of the launch, last thing: true (all threads) in the block that
// leaves last, which changes what the launch's guard is read from and resets
// the door (nobody looks at either any more).
__device__ __forceinline__ bool door_leave(Door *b, uint32_t blocks) {
  __shared__ int last;
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    last = bar_add(&b->gone) + 1 == blocks;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  return last != 0;
}

__device__ __forceinline__ void door_reset(Door *b) {
  uint32_t *count = &b->full[0][0];
  constexpr int kCounts = (int)((sizeof(b->full) + sizeof(b->group)) / sizeof(uint32_t));
  for (int i = threadIdx.x; i < kCounts; i += blockDim.x) count[i] = 0;
  if (threadIdx.x == 0) b->arrived = b->parts = b->gone = 0;
}

}  // namespace sc

#endif
