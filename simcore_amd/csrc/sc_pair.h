// sc_pair.h -- device code of one candidate pair, shared by the pair kernels
// (sc_pair.hip) and the step kernel that runs the pair pass and the
// integrator in one launch (sc_integrate_long.hip).  The two files are
// compiled with different contraction defaults; every function here states
// its own, so both produce the same bits.
#pragma once

#include <hip/hip_runtime.h>

#include "sc_internal.h"
#include "sc_math.h"

namespace sc {

// A bond as the pair pass uses it.  FP64 path: the scaled position, as
// Bond::ReInit stores it.  Mixed path: the position in cell units, cell
// index plus the record's 32-bit offset (exact in FP64), so that the
// separation of two bonds is an exact difference and one multiplication.
struct BondRec {
  double s[3], u[3], len;
};

template <bool MIXED>
__device__ __forceinline__ BondRec load_rec(const double *br, const Geo &g, int64_t b) {
  BondRec r;
  if (MIXED) {
#pragma clang fp contract(fast)
    const uint4 *rec = reinterpret_cast<const uint4 *>(br + 4 * b);
    const uint4 a = rec[0], v = rec[1];
    const int packed = (int)v.z;
    constexpr double k32 = 1.0 / 4294967296.0;
    r.s[0] = (double)(packed & 1023) + (double)a.x * k32;
    r.s[1] = (double)((packed >> 10) & 1023) + (double)a.y * k32;
    r.s[2] = (double)((packed >> 20) & 1023) + (double)a.z * k32;
    oct_decode(v.x, v.y, r.u);
    r.len = (double)__uint_as_float(a.w) + (double)__uint_as_float(v.w);
  } else {
    rec_read_full(br, b, r.s, r.u, &r.len);
  }
  return r;
}

// Mixed path: separation r2 - r1 of two cell-unit positions with the
// minimum-image rule of the reference's ds -= NINT(ds) (|ds| >= half the
// box wraps), times the cell length.
__device__ __forceinline__ void sep_cells(const Geo &g, const double *p1, const double *p2,
                                          double *sep) {
#pragma clang fp contract(fast)
  const double n = (double)g.n1d, half = 0.5 * (double)g.n1d;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double ds = p2[k] - p1[k];
    const double w = ds >= half ? ds - n : (ds <= -half ? ds + n : ds);
    sep[k] = w * (g.h[4 * k] * g.inv_n1d);
  }
}

// Mixed-precision MinimumDistance::Sphero (src/minimum_distance.cpp:231-343):
// the reference's FP64 arithmetic and branch rules, except that the division
// by 1-(u1.u2)^2 multiplies by the hardware FP32 reciprocal (relative error
// ~1e-7).  A clamped line parameter is recomputed exactly from the other
// one, so the reciprocal's error reaches only unclamped parameters
// (|lambda| <= l/2).  On CDNA4 an FP64 FMA issues at the rate of an
// unpacked FP32 one, so keeping the geometry in FP64 costs nothing and
// needs no separate near-parallel path; only the divisions and square roots
// (many instructions in IEEE FP64) are replaced.  Multiply-adds are fused
// (one rounding each); both owners of a pair still run the same
// instructions on the same inputs.
__device__ __forceinline__ void sphero_mixed(const double *dr, const double *u1, double hl1,
                                             const double *u2, double hl2, double *rmin,
                                             double *rm2, double *lam_o, double *mu_o) {
#pragma clang fp contract(fast)
  double a = 0.0, b = 0.0, c = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    a += dr[i] * u1[i];
    b += dr[i] * u2[i];
    c += u1[i] * u2[i];
  }
  double lambda, mu;
  const double denom = 1.0 - c * c;
  if (denom < 1.0e-12) {
    lambda = 0.5 * a;
    mu = -0.5 * b;
  } else {
    const double id = (double)__builtin_amdgcn_rcpf((float)denom);
    lambda = (a - c * b) * id;
    mu = (-b + c * a) * id;
  }
  const double lm = dabs(lambda), mm = dabs(mu);
  if (lm > hl1 && mm > hl2) {
    const double la = dsign(hl1, lambda);
    double ma = -b + la * c;
    if (dabs(ma) > hl2) ma = dsign(hl2, ma);
    const double mb = dsign(hl2, mu);
    double lb = a + mb * c;
    if (dabs(lb) > hl1) lb = dsign(hl1, lb);
    double m2a = 0.0, m2b = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double ra = dr[i] - la * u1[i] + ma * u2[i];
      const double rb = dr[i] - lb * u1[i] + mb * u2[i];
      m2a += ra * ra;
      m2b += rb * rb;
    }
    if (m2a < m2b) {
      lambda = la;
      mu = ma;
    } else {
      lambda = lb;
      mu = mb;
    }
  } else if (lm > hl1) {
    lambda = dsign(hl1, lambda);
    mu = -b + lambda * c;
    if (dabs(mu) > hl2) mu = dsign(hl2, mu);
  } else if (mm > hl2) {
    mu = dsign(hl2, mu);
    lambda = a + mu * c;
    if (dabs(lambda) > hl1) lambda = dsign(hl1, lambda);
  }
  double m2 = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    rmin[i] = dr[i] - lambda * u1[i] + mu * u2[i];
    m2 += rmin[i] * rmin[i];
  }
  *rm2 = m2;
  *lam_o = lambda;
  *mu_o = mu;
}

// WCA force of WCAPotential::CalcPotential (include/simcore/wca_potential.hpp:
// 14-32) with 1/r from the hardware FP32 reciprocal square root refined by
// one FP64 Newton step (relative error ~1e-14), rounded to FP32 for the
// slot.  dr^2 >= 1e-12 here.
__device__ __forceinline__ float4 wca_mixed(const Geo &g, const double *rmin, double rm2) {
#pragma clang fp contract(fast)
  double rinv = (double)__builtin_amdgcn_rsqf((float)rm2);
  rinv = rinv * (1.5 - 0.5 * rm2 * rinv * rinv);
  const double rinv2 = rinv * rinv;
  const double r6 = rinv2 * rinv2 * rinv2;
  double ffac = -(12.0 * g.c12 * r6 - 6.0 * g.c6) * r6 * rinv;
  if (dabs(ffac) > g.fcut) ffac = (ffac >= 0.0 ? 1.0 : -1.0) * g.fcut;
  const double sc = ffac * rinv;
  return make_float4((float)(sc * rmin[0]), (float)(sc * rmin[1]), (float)(sc * rmin[2]),
                     (float)(rm2 * rinv));
}

// The pair of incidence q {partner, role | written << 1 | owner << 2},
// computed with the candidate's own (obj1, obj2) orientation
// (src/interaction_manager.cpp:448-498): the incidence's slot copy updated
// when in range (and marked written), else the copy's force, 0 if it was
// not written since the rebuild (the reference's fresh pair record).  Both
// owners of a candidate run the same instructions on the same inputs and
// obtain the same bits, so their slot copies stay equal.  The slot's fourth
// value is the pair's signed distance (pair_force64): with the force it
// gives the pair's stress and potential energy, so the sticky record needs
// nothing else.  Returns the candidate's force in fc, the owner's contact
// parameter (lambda for obj1, mu for obj2) in *sc and the signed distance
// in *rs (0 for a slot not written since the rebuild).
template <bool MIXED>
__device__ __forceinline__ void pair_slot(const Dev &d, const Geo &g, const BondRec &own,
                                          int32_t q, int2 ent, const BondRec &oth, double *fc,
                                          double *sc, double *rs_out) {
#pragma clang fp contract(off)
  const bool second = (ent.y & 1) != 0;  // this bond is obj2 of the candidate
  const bool written = (ent.y & 2) != 0;
  // obj1 and obj2 by selection (no branch on the role)
  double u1[3], u2[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    u1[k] = second ? oth.u[k] : own.u[k];
    u2[k] = second ? own.u[k] : oth.u[k];
  }
  const double l1 = second ? oth.len : own.len;
  const double l2 = second ? own.len : oth.len;
  double lam, mu, rs = 0.0;
  fc[0] = fc[1] = fc[2] = 0.0;
  bool wrote = false;
  if (!MIXED) {
    double s1[3], s2[3], dr[3], dr2;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s1[k] = second ? oth.s[k] : own.s[k];
      s2[k] = second ? own.s[k] : oth.s[k];
    }
    sphero64(g.h, s1, u1, l1, s2, u2, l2, dr, &dr2, &lam, &mu);
    if (!(dr2 > g.rcut2)) {
      double f[3];
      if (pair_force64(g.c12, g.c6, g.fcut, dr, dr2, lam, mu, u1, u2, f, &rs)) {
        fc[0] = f[0];
        fc[1] = f[1];
        fc[2] = f[2];
        d.islot64[q] = make_double4(f[0], f[1], f[2], rs);
        wrote = true;
      }
    }
    if (!wrote && written) {
      const double4 o = d.islot64[q];
      fc[0] = o.x;
      fc[1] = o.y;
      fc[2] = o.z;
      rs = o.w;
    }
  } else {
    // obj2 - obj1: the owner-to-partner separation, negated for obj2 (the
    // minimum-image rule is odd, so both owners get the same bits)
    double sep[3], dr[3], dr2;
    sep_cells(g, own.s, oth.s, sep);
#pragma unroll
    for (int k = 0; k < 3; ++k) sep[k] = second ? -sep[k] : sep[k];
    sphero_mixed(sep, u1, 0.5 * l1, u2, 0.5 * l2, dr, &dr2, &lam, &mu);
    if (!(dr2 > g.rcut2)) {
      float4 f4;
      if (dr2 < 1.0e-12) {
        // MaxForcePotential branch (include/simcore/max_force_potential.hpp:
        // 11-40), FP64 as the reference; practically never taken
        double f[3];
        wrote = pair_force64(g.c12, g.c6, g.fcut, dr, dr2, lam, mu, u1, u2, f, &rs) != 0;
        f4 = make_float4((float)f[0], (float)f[1], (float)f[2], (float)rs);
      } else {
        f4 = wca_mixed(g, dr, dr2);
        wrote = true;
      }
      if (wrote) {
        d.islot32[q] = f4;
        fc[0] = f4.x;
        fc[1] = f4.y;
        fc[2] = f4.z;
        rs = f4.w;
      }
    }
    if (!wrote && written) {
      const float4 o = d.islot32[q];
      fc[0] = o.x;
      fc[1] = o.y;
      fc[2] = o.z;
      rs = o.w;
    }
  }
  *rs_out = rs;
  *sc = second ? mu : lam;
  if (wrote && !written) reinterpret_cast<int32_t *>(d.inc)[2 * (int64_t)q + 1] = ent.y | 2;
}

// The owner's share of a pair (src/interaction_manager.cpp:469-470,
// 500-517; src/minimum_distance.cpp:339-342): +F and contact1 x F for obj1,
// -F and -(contact2 x F) for obj2.  With f the signed force (-F for obj2)
// the torque is contact x f, the same bits as -(contact x F).  The mixed
// path fuses the cross product's multiply-adds.
template <bool MIXED>
__device__ __forceinline__ void pair_share(const double *u, double sc, const double *f,
                                           double *t) {
#pragma clang fp contract(off)
  double con[3];
  for (int k = 0; k < 3; ++k) con[k] = sc * u[k];
  if (MIXED) {
#pragma clang fp contract(fast)
    t[0] = con[1] * f[2] - con[2] * f[1];
    t[1] = con[2] * f[0] - con[0] * f[2];
    t[2] = con[0] * f[1] - con[1] * f[0];
  } else {
    cross3(con, f, t);
  }
}

// Per-bond sums, accumulated in FP64; FP32 storage on the mixed path (one
// rounding of the sum).
template <bool MIXED>
__device__ __forceinline__ void store_bond_sums(const Dev &d, int64_t nb, int64_t b,
                                                const double *F, const double *T) {
  for (int k = 0; k < 3; ++k) {
    if (MIXED) {
      d.bf32[k * nb + b] = (float)F[k];
      d.bt32[k * nb + b] = (float)T[k];
    } else {
      d.bf[k * nb + b] = F[k];
      d.bt[k * nb + b] = T[k];
    }
  }
}

}  // namespace sc
