// sc_limits.h -- how long the candidate lists may get, for the kernels that
// count them and the host code that allocates them, and up to which length the
// balanced pair kernel serves them.
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

// Mean length of a bond's list up to which the balanced pair kernel is the
// faster one.  Its lanes evaluate 128 entries and then each bond's lane adds
// up the bond's, so with long lists a few lanes add while the others wait;
// the per-bond kernel has every lane at its own list, all of about the same
// length, but needs enough bonds to fill the chip.  us a pass, balanced /
// per bond with 256 threads, by mean length: 4k bonds 65: 100 / 130, 151: 222
// / 260, 317: 425 / 424; 50k 64: 142 / 184, 100: 243 / 231; 100k 27: 111 / 144,
// 52: 204 / 189, 103: 473 / 303; 200k 35: 209 / 214, 52: 359 / 317; 600k 50:
// 717 / 806, 101: 1834 / 1580.  Just above 131072 bonds, where a wavefront
// takes 64 of them, they are too few to fill the chip: at 150k equal at 19 and
// 1.28 times the time at 32.  FP64's lines lie up to a fifth lower.
inline double longest_balanced(int64_t nb) {
  return nb <= 32768 ? 160.0 : nb <= 65536 ? 80.0 : nb <= 131072 ? 32.0 : nb < 200000 ? 16.0 : 40.0;
}

// Whether a system whose lists have `mean` entries a bond takes the balanced
// kernel; `now`: whether it does at present.  The lists have to get a quarter
// shorter again before the choice changes back.
inline bool pair_balanced(int64_t nb, double mean, bool now) {
  return mean <= longest_balanced(nb) * (now ? 1.0 : 0.75);
}

}  // namespace sc

#endif
