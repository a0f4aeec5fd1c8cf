// sc_thomas.h -- the FP64 integrator's Thomas solve and the division it
// shares between two quotients.  Everything here also compiles for the host,
// with the two hardware operations written out, so that the quotients can be
// compared with the host's divisions over the whole range of doubles.
#ifndef SIMCORE_AMD_THOMAS_H_
#define SIMCORE_AMD_THOMAS_H_

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>

namespace sc {

constexpr int kAhead = 2;  // rows loaded ahead of a chain (120 registers, four
                           // wavefronts per SIMD; 4 rows take 144)

__host__ __device__ __forceinline__ uint64_t double_bits(double x) {
  uint64_t b;
  __builtin_memcpy(&b, &x, sizeof(b));
  return b;
}

// v_rcp_f64 (the host's is exact where the hardware's is an estimate; two
// refinements follow either way)
__host__ __device__ __forceinline__ double rcp_estimate(double x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcp(x);
#else
  return 1.0 / x;
#endif
}

// v_div_fixup_f64, as the instruction set manual defines it: quotient q of
// num / den with the signs and special values of an IEEE division
__host__ __device__ __forceinline__ double div_fixup(double q, double den, double num) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_div_fixup(q, den, num);
#else
  const uint64_t kSign = 1ull << 63, sign = (double_bits(num) ^ double_bits(den)) & kSign;
  auto with_sign = [&](double v) {
    const uint64_t b = (double_bits(v) & ~kSign) | sign;
    std::memcpy(&v, &b, sizeof(v));
    return v;
  };
  const int en = (int)(double_bits(num) >> 52 & 2047), ed = (int)(double_bits(den) >> 52 & 2047);
  const double inf = __builtin_inf();
  if (num != num || den != den) return num + den;
  const bool ni = num == inf || num == -inf, di = den == inf || den == -inf;
  if ((num == 0 && den == 0) || (ni && di)) return __builtin_nan("");
  if (den == 0 || ni) return with_sign(inf);
  if (di || num == 0) return with_sign(0.0);
  if (en - ed < -1075) return with_sign(0.0);
  return with_sign(q);
#endif
}

// IEEE division of several numerators by one denominator: the refined
// reciprocal is shared and each quotient rounds once more, which gives the
// correctly rounded quotient (the steps of the hardware division sequence
// without its operand scaling).  81 clocks for two dependent quotients in a
// chain, against 138 for two IEEE divisions as the compiler expands them (one
// wavefront, measured).
//
// Without the scaling no intermediate value may leave the normal range, so
// this holds for |den| in [2^-150, 2^100], |num| zero or at least kLeastShared
// and a finite quotient; div_fixup supplies zeros, infinities and NaNs.
//   den: the pivots of a solve.  The matrices are the projections of positive
//     definite ones on the bonds, whose eigenvalues lie between the smallest
//     friction's and a few times the largest, less a factor of (sites)^2 =
//     2^16.  shared_frictions() bounds the frictions and their ratio, so the
//     pivots lie between 2^-90 and 2^55, far from where rounding could cancel
//     them.
//   num: small ones are caught by thomas_chain as they come.  A quotient that
//     overflows leaves an infinity or a NaN (the remainder of an infinite
//     quotient is a NaN, where the IEEE division has an infinity), which
//     every later row passes on, so the last row's value tells.
constexpr double kLeastShared = 0x1p-900;

__host__ __device__ __forceinline__ bool shared_frictions(double gpar, double gperp) {
  return gpar > 0x1p-50 && gpar < 0x1p50 && gperp > 0x1p-50 && gperp < 0x1p50 &&
         gpar < gperp * 0x1p20 && gperp < gpar * 0x1p20;
}

__host__ __device__ __forceinline__ double shared_rcp(double den) {
  double y = rcp_estimate(den);
  y = __builtin_fma(y, __builtin_fma(-den, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-den, y, 1.0), y);
}
__host__ __device__ __forceinline__ double shared_quot(double num, double den, double y) {
  const double m = num * y;
  return div_fixup(__builtin_fma(__builtin_fma(-den, m, num), y, m), den, num);
}

// e with 2^(e-1) <= |x| < 2^e, subnormal x too; 0 for zero, infinities and NaN
// (v_frexp_exp_i32_f64), so a minimum over numerators ignores those
__host__ __device__ __forceinline__ int exponent_of(double x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_frexp_exp(x);
#else
  int e = 0;
  if (x - x == 0.0) (void)std::frexp(x, &e);
  return e;
#endif
}
constexpr int kLeastExponent = -899;  // of kLeastShared

// Thomas with the reference's operation order on symmetric rows {diagonal,
// right-hand side} and off-diagonals off[i] (rows i, i+1); the solution
// replaces the right-hand side.  `rows` is the same for every lane: rows
// past a filament's last are {1, 0} with off-diagonal 0, which solve to 0
// and leave the others as they are, so no lane needs a branch.  The last row's
// solution is the forward recursion's value there.  FAST: quotients by
// shared_quot; returns false when a numerator was out of its range (the
// caller then sets the rows up again and takes the plain divisions).
template <bool FAST>
__host__ __device__ __forceinline__ bool thomas_chain(int rows, double2 *row, const double *off) {
  int least = 0;
  double cp = 0.0, dp = 0.0, lo = 0.0;
  double2 v[kAhead];
  double c[kAhead];
  auto load = [&](int i0) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int i = i0 + k < rows ? i0 + k : rows - 1;
      v[k] = row[i];
      c[k] = off[i];
    }
  };
  auto step = [&](int i, const double2 &w, double o) {
    const double den = w.x - lo * cp;  // (row 0: lo, cp and dp are 0)
    const double num = w.y - lo * dp;
    if (FAST) {
      const double y = shared_rcp(den);
      const int e = exponent_of(num);
      least = e < least ? e : least;
      cp = shared_quot(o, den, y);
      dp = shared_quot(num, den, y);
    } else {
      cp = o / den;
      dp = num / den;
    }
    lo = o;
    row[i] = make_double2(cp, dp);
  };
  load(0);
  int i0 = 0;
  for (; i0 + kAhead <= rows; i0 += kAhead) {
    double2 w[kAhead];
    double o[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      w[k] = v[k];
      o[k] = c[k];
    }
    load(i0 + kAhead);
#pragma unroll
    for (int k = 0; k < kAhead; ++k) step(i0 + k, w[k], o[k]);
  }
#pragma unroll
  for (int k = 0; k < kAhead; ++k)
    if (i0 + k < rows) step(i0 + k, v[k], c[k]);
  // back substitution, rows rows-2 .. 0
  const double last = dp;  // infinite or NaN if any quotient was
  double x = dp;
  auto loadb = [&](int j0) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) v[k] = row[j0 - k > 0 ? j0 - k : 0];
  };
  int j0 = rows - 2;
  loadb(j0);
  for (; j0 - kAhead + 1 >= 0; j0 -= kAhead) {
    double2 w[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) w[k] = v[k];
    loadb(j0 - kAhead);
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      x = w[k].y - w[k].x * x;
      row[j0 - k].y = x;
    }
  }
#pragma unroll
  for (int k = 0; k < kAhead; ++k)
    if (j0 - k >= 0) {
      x = v[k].y - v[k].x * x;
      row[j0 - k].y = x;
    }
  return !FAST || (least >= kLeastExponent && last - last == 0.0);
}

}  // namespace sc

#endif
