// sc_integrate.hip -- Filament::UpdatePosition (src/filament.cpp:394-428) on
// the FP64 path: every operation in the reference's order, so the results are
// those of the CPU path bit for bit.
//
// Mapping: one site per lane.  A block of 256 lanes holds as many filaments
// of one length bin as fit (the bin's longest filament sets the slice), and
// one launch serves every bin, the longest first, so that their chains run
// beside the short filaments' instead of after them.  Per-site values live in
// LDS, one slice per filament, odd strides between slices.
//
// The reference's sequential pieces -- the two Thomas solves
// (src/linear_algebra.cpp:164-197), the metric-determinant recursions
// (src/filament.cpp:613-623) and bond renormalisation (:904-924) -- run one
// filament per lane of one wavefront, the recursion in registers and the
// coefficients of the next rows loaded from LDS while the current ones are
// worked on; a midstep's determinant recursions run in a second wavefront
// beside its random-force solve.
//
// Bound: the latency of those chains (about 100 clocks a Thomas row, most of
// it the division) and, for large systems, instruction issue.  Measured, full
// step and midstep: 925 x 8 filaments of 8-256 sites (229k bonds) 52 and 64 us
// where the six launches, one per bin, with chains branching and loading row
// by row took 190 and 260; 5000 filaments of 32 sites 27 and 29 us (31, 40).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sc_internal.h"
#include "sc_math.h"
#include "sc_thomas.h"

namespace sc {

namespace {

constexpr int kExactBlock = 256;
constexpr int kSlots = 288;    // site slots of a block: slices of odd stride
constexpr int kMaxChains = 64;  // filaments of a block: one lane each in a chain

// Slice layout of filaments of at most w sites: the stride between slices
// (odd, so that the chains' lanes, one per slice, hit different banks) and
// how many fit a block.
__host__ __device__ __forceinline__ int exact_stride(int w) { return w | 1; }
__host__ __device__ __forceinline__ int exact_per_block(int w) {
  const int a = kExactBlock / w, b = kSlots / exact_stride(w);
  const int n = a < b ? a : b;
  return n < kMaxChains ? (n < 1 ? 1 : n) : kMaxChains;
}

// Metric determinants (src/filament.cpp:613-623) from the cosines cs[0..n-3]
// of n sites: det_t[0..rows-1] forward from the tail (entries past n-1 are
// not used)
__device__ __forceinline__ void det_tail(int rows, const double *cs, double *dt) {
  double t2 = 1.0, t1 = 2.0;
  dt[0] = 1;
  dt[1] = 2;
  double f[kAhead];
  auto load = [&](int i0) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) f[k] = cs[(i0 + k < rows ? i0 + k : rows - 1) - 2];
  };
  load(2);
  for (int i0 = 2; i0 < rows; i0 += kAhead) {
    double w[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) w[k] = f[k];
    load(i0 + kAhead);
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
      if (i0 + k < rows) {
        const double v = 2 * t1 - (-w[k]) * (-w[k]) * t2;
        dt[i0 + k] = v;
        t2 = t1;
        t1 = v;
      }
  }
}

// det_b[j], kept at db[j-1] for j = 1..n, backward from the head; `rows` is
// the block's, lanes of shorter filaments run out of entries and write to
// their slice's spare slot db[spare]
__device__ __forceinline__ void det_head(int rows, int n, const double *cs, double *db,
                                         int spare) {
  double b2 = 1.0, b1 = 2.0;
  db[n - 1] = 1;
  db[n - 2] = 2;
  double f[kAhead];
  auto load = [&](int i0) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int j = n - 1 - (i0 + k);
      f[k] = cs[j >= 0 ? j : 0];
    }
  };
  load(2);
  for (int i0 = 2; i0 < rows; i0 += kAhead) {
    double w[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) w[k] = f[k];
    load(i0 + kAhead);
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
      if (i0 + k < rows) {
        const double v = 2 * b1 - (-w[k]) * (-w[k]) * b2;
        const int j = n - 1 - (i0 + k);
        db[j >= 0 ? j : spare] = v;
        b2 = b1;
        b1 = v;
      }
  }
}

}  // namespace

__global__ __launch_bounds__(kExactBlock) void k_integrate_exact(Dev d, Geo g, ExactBins eb) {
  // (an aborted step leaves every lane inactive rather than returning: the
  // list and site loads then need not wait for the control block)
  const bool live = d.ctl->abort == 0;
  // the block's bin (uniform)
  int bin = 0;
#pragma unroll
  for (int k = 1; k < kMaxBins; ++k)
    if (k < eb.n && (int)blockIdx.x >= eb.blk0[k]) bin = k;
  const int4 *list = eb.list[0];
  int count = eb.count[0], w = eb.width[0], blk0 = eb.blk0[0];
#pragma unroll
  for (int k = 1; k < kMaxBins; ++k)
    if (k == bin) {
      list = eb.list[k];
      count = eb.count[k];
      w = eb.width[k];
      blk0 = eb.blk0[k];
    }
  const int per = exact_per_block(w), stride = exact_stride(w);
  const int t = threadIdx.x;
  const int grp = t / w, i = t - grp * w;  // the lane's filament and site
  const int fidx = ((int)blockIdx.x - blk0) * per + grp;
  const bool listed = grp < per && fidx < count, active = listed && live;
  const int4 ent = listed ? list[fidx] : make_int4(0, 0, 0, 0);
  const int f = ent.x, n = live ? ent.z : 0;
  const int64_t s0 = ent.y;
  const int64_t b0 = s0 - f;
  const int64_t ns = g.ns, nb = g.nb;
  const bool mid = step_is_mid(d);
  const int64_t step = step_index(d);
  double bl = 1.0, kappa = 0.0, gpar = 1.0, gperp = 1.0, sgpar = 0.0, sgperp = 0.0;
  if (active) {
    const double *fp = d.fpar + 8 * f;
    bl = fp[0];
    kappa = fp[1];
    gpar = fp[2];
    gperp = fp[3];
    sgpar = fp[4];
    sgperp = fp[5];
  }

  __shared__ double U_[3][kSlots], F_[3][kSlots], T_[3][kSlots], R_[3][kSlots];
  __shared__ double2 P_[kSlots];  // rows of a solve: {diagonal, right-hand side}
  __shared__ double C_[kSlots], CS_[kSlots];
  __shared__ double sbl[kMaxChains];
  __shared__ int sn[kMaxChains], sfil[kMaxChains], sbad[kMaxChains], slow;
  const int at = active ? grp * stride : 0;  // the filament's slice
  double *U[3] = {U_[0] + at, U_[1] + at, U_[2] + at};
  double *FS[3] = {F_[0] + at, F_[1] + at, F_[2] + at};  // site forces, then new orientations
  double *TN[3] = {T_[0] + at, T_[1] + at, T_[2] + at};  // bond torque terms, then tangents
  // bond force halves; random forces; determinants and K_eff; new positions
  double *RR[3] = {R_[0] + at, R_[1] + at, R_[2] + at};
  double2 *P = P_ + at;
  double *CS = CS_ + at;
  const bool site = i < n, bond = i < n - 1;
  // the lane's row of a solve: row, unit row past the last, or none
  const bool slot = grp < per;
  const int row = grp * stride + i;
  const bool sane = shared_frictions(gpar, gperp);

  // ---- loads -------------------------------------------------------------
  double rp_reg[3], fr[3] = {0.0, 0.0, 0.0}, u[3] = {0.0, 0.0, 0.0};
  double Fb[3], Tb[3];
  if (i == 0 && grp < per && grp < kMaxChains) {
    sn[grp] = n;
    sfil[grp] = f;
    sbl[grp] = bl;
    sbad[grp] = 0;
  }
  if (t == 0) slow = 0;
  if (site) {
    for (int q = 0; q < 3; ++q) rp_reg[q] = mid ? d.r[q * ns + s0 + i] : d.rp[q * ns + s0 + i];
    // the last site takes the last bond's orientation
    double rs[3], rl;
    rec_read_full(d.br, b0 + (bond ? i : n - 2), rs, u, &rl);
    if (bond)
      for (int q = 0; q < 3; ++q) {
        Fb[q] = d.bf[q * nb + b0 + i];
        Tb[q] = d.bt[q * nb + b0 + i];
      }
    for (int q = 0; q < 3; ++q) U[q][i] = u[q];
    if (!mid && g.stoch)
      for (int q = 0; q < 3; ++q) fr[q] = d.fr[q * ns + s0 + i];
  }
  // ---- ApplyInteractionForces (src/filament.cpp:992-1048) ----------------
  // per bond: F/2 into RR, (u x T)/l into TN (TN is rebuilt below)
  const double linv = 1.0 / bl;
  if (bond) {
    double pt[3];
    cross3(u, Tb, pt);
    for (int q = 0; q < 3; ++q) {
      TN[q][i] = pt[q] * linv;
      RR[q][i] = 0.5 * Fb[q];
    }
  }
  __syncthreads();
  double fs[3] = {0.0, 0.0, 0.0}, um[3] = {0.0, 0.0, 0.0}, up[3] = {0.0, 0.0, 0.0};
  double tg[3] = {0.0, 0.0, 0.0};
  if (site) {
    if (i >= 1) {
      for (int q = 0; q < 3; ++q) um[q] = U[q][i - 1];
      for (int q = 0; q < 3; ++q) fs[q] += RR[q][i - 1];
      for (int q = 0; q < 3; ++q) fs[q] += -TN[q][i - 1];
    }
    if (i <= n - 2) {
      for (int q = 0; q < 3; ++q) up[q] = U[q][i + 1];
      for (int q = 0; q < 3; ++q) fs[q] += RR[q][i];
      for (int q = 0; q < 3; ++q) fs[q] += TN[q][i];
    }
    // ---- CalculateAngles / CalculateTangents -----------------------------
    if (i < n - 2) CS[i] = dot3(u, up);
    if (i == 0 || i == n - 1) {
      for (int q = 0; q < 3; ++q) tg[q] = u[q];  // the end bond's (see the loads)
    } else {
      for (int q = 0; q < 3; ++q) tg[q] = um[q] + u[q];
      normalize3(tg);
    }
  }
  __syncthreads();
  if (site)
    for (int q = 0; q < 3; ++q) TN[q][i] = tg[q];

  // ---- random forces (midstep) -------------------------------------------
  const bool draws = mid && g.stoch;
  if (draws && site) {
    // ConstructUnprojectedRandomForces (src/filament.cpp:518-548)
    double xi[3], xt[3];
    draw_xi(g, (int64_t)d.noise_off[f] + i, (step - 1) >> 1, xi);
    const double t0 = tg[0], t1 = tg[1], t2 = tg[2];
    xt[0] = t0 * t0 * xi[0] + t0 * t1 * xi[1] + t0 * t2 * xi[2];
    xt[1] = t1 * t1 * xi[1] + t0 * t1 * xi[0] + t1 * t2 * xi[2];
    xt[2] = t2 * t2 * xi[2] + t0 * t2 * xi[0] + t1 * t2 * xi[1];
    for (int q = 0; q < 3; ++q) {
      fr[q] = sgperp * xi[q] + (sgpar - sgperp) * xt[q];
      RR[q][i] = fr[q];
    }
  }
  __syncthreads();
  // GeometricallyProjectRandomForces (src/filament.cpp:550-599)
  auto set_row = [&](double diag, double rhs, double off) {
    P_[row] = make_double2(diag, rhs);
    C_[row] = off;
    if (!sane || (off != 0.0 && dabs(off) < kLeastShared)) slow = 1;
  };
  double rhs = 0.0;
  if (draws && slot) {
    double tmp[3] = {0.0, 0.0, 0.0}, off = 0.0;
    if (bond) {
      for (int q = 0; q < 3; ++q) tmp[q] = RR[q][i + 1] - fr[q];
      rhs = dot3(tmp, u);
      if (i < n - 2) off = -CS[i];
    }
    set_row(bond ? 2.0 : 1.0, rhs, off);
  }
  __syncthreads();
  // one filament per lane: the random-force solve in the first wavefront, the
  // determinants (into R_[0], R_[1], whose random forces are in registers by
  // now) in the second and third
  const int chain = t & 63, cw = t >> 6;
  const bool runs = chain < per, fils = runs && sn[chain] > 0;
  const int o = chain * stride;
  if (cw == 0 && draws && runs && !thomas_chain<true>(w, P_ + o, C_ + o)) slow = 1;
  if (cw == 1 && runs) det_tail(w, CS_ + o, R_[0] + o);
  if (cw == 2 && fils) det_head(w, sn[chain], CS_ + o, R_[1] + o, stride - 1);
  __syncthreads();
  if (draws && slow) {  // numbers shared_quot does not serve
    if (slot) {
      P_[row] = make_double2(bond ? 2.0 : 1.0, rhs);
      C_[row] = i < n - 2 ? -CS[i] : 0.0;
    }
    __syncthreads();
    if (t == 0) slow = 0;
    if (cw == 0 && runs) thomas_chain<false>(w, P_ + o, C_ + o);
    __syncthreads();
  }
  if (mid && site) {
    if (draws) {
      double p[3];
      if (i == 0) {
        for (int q = 0; q < 3; ++q) p[q] = fr[q] + P[0].y * u[q];
      } else if (i == n - 1) {
        for (int q = 0; q < 3; ++q) p[q] = fr[q] - P[n - 2].y * u[q];
      } else {
        for (int q = 0; q < 3; ++q) p[q] = fr[q] + P[i].y * u[q] - P[i - 1].y * um[q];
      }
      for (int q = 0; q < 3; ++q) {
        d.fr[q * ns + s0 + i] = p[q];
        fr[q] = p[q];
      }
    }
    // Mesh::UpdatePrevPositions (src/mesh.cpp:175-182)
    for (int q = 0; q < 3; ++q) d.rp[q * ns + s0 + i] = rp_reg[q];
  }
  // AddRandomForces (src/filament.cpp:601-606)
  if (g.stoch && site)
    for (int q = 0; q < 3; ++q) fs[q] += fr[q];

  // ---- CalculateBendingForces, 3D (src/filament.cpp:608-776) -------------
  double *KE = RR[2];
  if (i < n - 2) {
    const double ginv = CS[i] * RR[0][i] * RR[1][i + 2] / RR[0][n - 1];
    KE[i] = (kappa + bl * ginv) / (bl * bl);
  }
  __syncthreads();
  if (site) {
    double f3[3] = {0.0, 0.0, 0.0};
    if (i > 1) {
      double u1[3] = {U[0][i - 2], U[1][i - 2], U[2][i - 2]};
      bend_add(f3, KE[i - 2], u1, um);
    }
    if (i > 0 && i < n - 1) bend_mid(f3, KE[i - 1], um, u);
    if (i < n - 2) bend_sub(f3, KE[i], u, up);
    for (int q = 0; q < 3; ++q) {
      fs[q] += f3[q];
      FS[q][i] = fs[q];
    }
  }
  __syncthreads();

  // ---- CalculateTensions (src/filament.cpp:778-838) ----------------------
  const double igpar = 1.0 / gpar, igperp = 1.0 / gperp;
  double diag = 1.0, off = 0.0;
  rhs = 0.0;
  if (bond) {
    double t2[3] = {TN[0][i + 1], TN[1][i + 1], TN[2][i + 1]};
    double f2[3] = {FS[0][i + 1], FS[1][i + 1], FS[2][i + 1]};
    double fd[3];
    for (int a = 0; a < 3; ++a) {
      double ta_ = gam(igpar, igperp, tg, a, 0) * fs[0] + gam(igpar, igperp, tg, a, 1) * fs[1];
      ta_ += gam(igpar, igperp, tg, a, 2) * fs[2];
      double tb_ = gam(igpar, igperp, t2, a, 0) * f2[0] + gam(igpar, igperp, t2, a, 1) * f2[1];
      tb_ += gam(igpar, igperp, t2, a, 2) * f2[2];
      fd[a] = tb_ - ta_;
    }
    rhs = dot3(u, fd);
    const double a1 = dot3(tg, u), a2 = dot3(t2, u);
    // 2 / gperp is 2 (1 / gperp), -1 / gperp is -(1 / gperp): the same bits
    diag = 2.0 * igperp + (igpar - igperp) * (a1 * a1 + a2 * a2);
    // the coupling of bonds i and i+1, row i+1's (src/filament.cpp:811-818)
    if (i < n - 2) off = -igperp * dot3(up, u) - (igpar - igperp) * (dot3(t2, u) * dot3(t2, up));
  }
  if (slot) set_row(diag, rhs, off);
  __syncthreads();
  if (cw == 0 && runs && !thomas_chain<true>(w, P_ + o, C_ + o)) slow = 1;
  __syncthreads();
  if (slow) {
    if (slot) {
      P_[row] = make_double2(diag, rhs);
      C_[row] = off;
    }
    __syncthreads();
    if (cw == 0 && runs) thomas_chain<false>(w, P_ + o, C_ + o);
    __syncthreads();
  }
  const double ti = bond ? P[i].y : 0.0, tl = i >= 1 && site ? P[i - 1].y : 0.0;
  if (bond) d.tension[b0 + i] = ti;

  // ---- UpdateSitePositions (src/filament.cpp:840-927) --------------------
  const double delta = mid ? 0.5 * g.delta : g.delta;
  double rn[3] = {0.0, 0.0, 0.0};
  if (site) {
    double f3[3] = {fs[0], fs[1], fs[2]};
    if (i == 0) {
      for (int q = 0; q < 3; ++q) f3[q] += ti * u[q];
    } else if (i == n - 1) {
      for (int q = 0; q < 3; ++q) f3[q] += -tl * u[q];
    } else {
      for (int q = 0; q < 3; ++q) f3[q] += ti * u[q] - tl * um[q];
    }
    for (int a = 0; a < 3; ++a) {
      double ft = gam(igpar, igperp, tg, a, 0) * f3[0] + gam(igpar, igperp, tg, a, 1) * f3[1];
      ft += gam(igpar, igperp, tg, a, 2) * f3[2];
      rn[a] = rp_reg[a] + delta * ft;
      RR[a][i] = rn[a];
    }
  }
  __syncthreads();
  // new lengths and orientations, CheckBondLengths (src/filament.cpp:934-951)
  double rd[3] = {0.0, 0.0, 0.0}, mm = 0.0;
  if (bond) {
    for (int q = 0; q < 3; ++q) {
      rd[q] = RR[q][i + 1] - rn[q];
      mm += rd[q] * rd[q];
    }
    mm = sqrt(mm);
    for (int q = 0; q < 3; ++q) {
      u[q] = rd[q] / mm;
      FS[q][i] = u[q];
    }
    const double diff = bl - mm;
    const double err = (diff < 0 ? -diff : diff) / bl;
    if (err > 1e-3) sbad[grp] = 1;
  }
  __syncthreads();
  if (cw == 0 && fils) {
    const int cf = sfil[chain], cn = sn[chain];
    int32_t sw = d.norm[2 * cf], nn = d.norm[2 * cf + 1];
    if (sbad[chain]) {
      sw = !sw;
      nn = 0;
      const double cbl = sbl[chain];
      double *X = R_[0] + o, *Y = R_[1] + o, *Z = R_[2] + o;
      const double *ux = F_[0] + o, *uy = F_[1] + o, *uz = F_[2] + o;
      if (sw) {
        double x = X[0], y = Y[0], z = Z[0];
#pragma unroll 4
        for (int k = 1; k < cn; ++k) {
          x = x + cbl * ux[k - 1];
          y = y + cbl * uy[k - 1];
          z = z + cbl * uz[k - 1];
          X[k] = x;
          Y[k] = y;
          Z[k] = z;
        }
      } else {
        double x = X[cn - 1], y = Y[cn - 1], z = Z[cn - 1];
#pragma unroll 4
        for (int k = cn - 1; k > 0; --k) {
          x = x - cbl * ux[k - 1];
          y = y - cbl * uy[k - 1];
          z = z - cbl * uz[k - 1];
          X[k - 1] = x;
          Y[k - 1] = y;
          Z[k - 1] = z;
        }
      }
    }
    nn++;
    d.norm[2 * cf] = sw;
    d.norm[2 * cf + 1] = nn;
  }
  __syncthreads();

  // ---- write back sites, Mesh::UpdateBondPositions, rebuild bookkeeping --
  double lmax = 0.0;
  if (site) {
    const bool moved = sbad[grp] != 0;
    if (moved)
      for (int q = 0; q < 3; ++q) rn[q] = RR[q][i];
    for (int q = 0; q < 3; ++q) d.r[q * ns + s0 + i] = rn[q];
    if (bond) {
      if (moved) {
        double r2[3] = {RR[0][i + 1], RR[1][i + 1], RR[2][i + 1]};
        bond_reinit(d, g, b0 + i, rn, r2, SC_PREC_FP64);
      } else {
        // the length and orientation bond_reinit would compute again
        double pos[3], sp[3];
        for (int q = 0; q < 3; ++q) pos[q] = rn[q] + 0.5 * rd[q];
        for (int k = 0; k < 3; ++k) {
          double si = 0.0;
          for (int j = 0; j < 3; ++j) si += g.hinv[3 * k + j] * pos[j];
          si -= (double)nint(si);
          sp[k] = si;
        }
        double4 *rec = reinterpret_cast<double4 *>(d.br_out + 8 * (b0 + i));
        rec[0] = make_double4(sp[0], sp[1], sp[2], u[0]);
        rec[1] = make_double4(u[1], u[2], mm, 0.0);
      }
    }
    if (!mid) {
      // Mesh::UpdateDrTot for the next step's rebuild test, two
      // Object::UpdateDrTot calls per site (src/mesh.cpp:533-544,
      // src/object.cpp:274-287)
      double a = d.acc[s0 + i];
      d.acc_prev[s0 + i] = a;
      for (int rep = 0; rep < 2; ++rep)
        for (int q = 0; q < 3; ++q) {
          const double dd = rn[q] - d.dr0[q * ns + s0 + i];
          a += dd * dd;
        }
      d.acc[s0 + i] = a;
      lmax = a;
    }
  }
  if (!mid) {
    for (int o = 32; o > 0; o >>= 1) {
      const double y = __shfl_xor(lmax, o, 64);
      lmax = y > lmax ? y : lmax;
    }
    if ((t & 63) == 0)
      atomicMax(&d.dr_slots[((int)blockIdx.x * (kExactBlock / 64) + (t >> 6)) & (kDrSlots - 1)],
                (unsigned long long)__double_as_longlong(lmax));
  }
}

void launch_integrate_exact(const Dev &d, const Geo &g, const BinDesc *bins, int n,
                            hipStream_t st) {
  // longest bin first
  int order[kMaxBins];
  ExactBins eb{};
  for (int k = 0; k < n && eb.n < kMaxBins; ++k)
    if (bins[k].count > 0) order[eb.n++] = k;
  std::sort(order, order + eb.n, [&](int a, int b) { return bins[a].maxn > bins[b].maxn; });
  int blocks = 0;
  for (int k = 0; k < eb.n; ++k) {
    const BinDesc &b = bins[order[k]];
    eb.list[k] = b.entries;
    eb.count[k] = b.count;
    eb.width[k] = b.width > 0 ? b.width : b.maxn;
    eb.blk0[k] = blocks;
    const int per = exact_per_block(eb.width[k]);
    blocks += (b.count + per - 1) / per;
  }
  if (blocks > 0)
    hipLaunchKernelGGL(k_integrate_exact, dim3((unsigned)blocks), dim3(kExactBlock), 0, st, d, g,
                       eb);
}

void launch_integrate(const Dev &d, const Geo &g, const BinDesc &bin, int precision,
                      const Tune &t, bool mid, hipStream_t st) {
  if (bin.count <= 0) return;
  if (precision == SC_PREC_FP64) {
    launch_integrate_exact(d, g, &bin, 1, st);
    return;
  }
  // mixed precision: register-resident variants
  if (launch_integrate_long(d, g, bin.list, bin.count, bin.maxn, precision, t.int_waves,
                            t.int_layout, mid, st))
    return;
  (void)launch_integrate_reg(d, g, bin.list, bin.count, bin.maxn, precision, t.int_waves, st);
}

}  // namespace sc
