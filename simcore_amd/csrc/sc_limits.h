// sc_limits.h -- how long the candidate lists may get, for the kernels that
// count them and the host code that allocates them.
#ifndef SIMCORE_AMD_LIMITS_H_
#define SIMCORE_AMD_LIMITS_H_

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace sc {

// Candidates are numbered in int32 and each incidence entry holds a
// candidate index shifted left by one bit; two entries a candidate.
constexpr int64_t kMaxCandidates = ((int64_t)1 << 30) - 1;

// A sum of list lengths kept in 32 bits.  Many bonds in few cells have lists
// whose sum passes 2^31 (1024 bonds of 2.1M entries); it is cut off at a
// length that no list may have, so that the total is still refused.
__host__ __device__ __forceinline__ int32_t kept_length(int64_t n) {
  return n > INT32_MAX ? INT32_MAX : (int32_t)n;
}
static_assert(INT32_MAX > 2 * kMaxCandidates, "a cut-off length does not fit");

// Candidates behind `total` entries (a cut-off one rounds up, past the limit).
__host__ __device__ __forceinline__ int64_t candidates_of(int64_t total) { return (total + 1) / 2; }

// Capacity after an overflow that asked for `need` candidates: doubled, or
// need + 25% + 1024 if more, at most kMaxCandidates unless need itself is
// larger (which the allocation then refuses).
inline int64_t grown_capacity(int64_t cap, int64_t need) {
  const int64_t want = std::max<int64_t>(2 * cap, need + need / 4 + 1024);
  return need > kMaxCandidates ? need : std::min(want, kMaxCandidates);
}

}  // namespace sc

#endif
