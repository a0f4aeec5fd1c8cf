// The limits by list length on the host, for test_list_limits.py.
#include "sc_limits.h"

extern "C" {

int64_t max_candidates() { return sc::kMaxCandidates; }
int32_t kept_length(int64_t n) { return sc::kept_length(n); }
int64_t candidates_of(int64_t total) { return sc::candidates_of(total); }
int64_t grown_capacity(int64_t cap, int64_t need) { return sc::grown_capacity(cap, need); }
int pair_balanced(int64_t nb, double mean, int now) { return sc::pair_balanced(nb, mean, now != 0); }

}  // extern "C"
