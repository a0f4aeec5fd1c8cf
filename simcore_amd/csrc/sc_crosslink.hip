// sc_crosslink.hip -- harmonic crosslinks between bonds.
//
// Force law and application: Crosslink::CalculateTetherForces
// (src/crosslink.cpp:246-273) with MinimumDistance::PointPoint
// (src/minimum_distance.cpp:71-101) between anchor points placed by
// Anchor::UpdateAnchorPositionToBond (src/anchor.cpp:236-248); torques of
// Anchor::ApplyAnchorForces (src/anchor.cpp:132-146).  Even steps recompute
// the forces (k_xl_force); every step the pair kernel adds the stored
// forces to the bonds first, in crosslink order, from per-bond lists
// {crosslink << 1 | anchor} sorted by crosslink (the reference's serial
// application order, src/crosslink_species.cpp:262-266).  Rebinding events
// (k_xl_events, even steps) and the list rebuild they trigger run after the
// pair kernel; the lists are rebuilt only when an event happened
// (Ctl::xl_dirty), on the device, so the step stays graph-replayable.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sc_block.h"
#include "sc_internal.h"
#include "sc_math.h"

namespace sc {

namespace {

// anchor point, orientation and length of bond b from its sites, with the
// arithmetic of Bond::ReInit (src/bond.cpp:22-37)
__device__ __forceinline__ void anchor_point(const Dev &d, const Geo &g, int32_t b, double lam,
                                             double *P, double *u, double *len) {
  const int64_t site = (int64_t)b + d.bond_fil[b];
  const int64_t ns = g.ns;
  double o[3], l = 0.0, pos[3];
  for (int k = 0; k < 3; ++k) {
    o[k] = d.r[k * ns + site + 1] - d.r[k * ns + site];
    l += o[k] * o[k];
  }
  l = sqrt(l);
  for (int k = 0; k < 3; ++k) {
    pos[k] = d.r[k * ns + site] + 0.5 * o[k];
    o[k] /= l;
  }
  for (int k = 0; k < 3; ++k) {
    u[k] = o[k];
    P[k] = pos[k] - (0.5 * l - lam) * u[k];
  }
  *len = l;
}

__device__ __forceinline__ void scaled(const Geo &g, const double *P, double *sp) {
  for (int i = 0; i < 3; ++i) {
    double si = 0.0;
    for (int j = 0; j < 3; ++j) si += g.hinv[3 * i + j] * P[j];
    si -= (double)nint(si);
    sp[i] = si;
  }
}

// scaled centre, orientation and length of bond b from its sites with the
// arithmetic of the FP64 bond record (Bond::ReInit + Object::UpdatePeriodic,
// src/bond.cpp:22-37, src/object.cpp:202-210): the partner search reads
// these rather than the record, which on the mixed path is compact (FP32)
__device__ __forceinline__ void bond_state(const Dev &d, const Geo &g, int32_t b, double *sp,
                                           double *u, double *len) {
  const int64_t site = (int64_t)b + d.bond_fil[b];
  const int64_t ns = g.ns;
  double o[3], l = 0.0, pos[3];
  for (int k = 0; k < 3; ++k) {
    o[k] = d.r[k * ns + site + 1] - d.r[k * ns + site];
    l += o[k] * o[k];
  }
  l = sqrt(l);
  for (int k = 0; k < 3; ++k) {
    pos[k] = d.r[k * ns + site] + 0.5 * o[k];
    u[k] = o[k] / l;
  }
  *len = l;
  scaled(g, pos, sp);
}

__device__ __forceinline__ double unit_draw(uint32_t v) {
  return ((double)v + 0.5) * 2.3283064365386962890625e-10;
}

// Crosslink forces: two lanes a crosslink, one per anchor, which exchange
// the scaled anchor points and each compute the same force and their own
// torque.  A chain of loads, FP64 roots and divisions bounds it, so the lanes
// halve it and small blocks spread it over the chip.
// 50k crosslinks: 8.6 us with one lane each, 7.8 with two.
constexpr int kXlBlock = 64;

__global__ __launch_bounds__(kXlBlock) void k_xl_force(Dev d, Geo g) {
  if (d.ctl->abort) return;
  const int64_t e = (int64_t)blockIdx.x * kXlBlock + threadIdx.x;
  if (e >= 2 * g.nx) return;
  const int a = (int)(e & 1);
  const double lam = d.xlam[e];
  double P[3], u[3], len, sp[3];
  anchor_point(d, g, d.xb[e], lam, P, u, &len);
  scaled(g, P, sp);
  double ds[3], dr[3], dr2 = 0.0;
  for (int i = 0; i < 3; ++i) {
    const double other = __shfl_xor(sp[i], 1);
    ds[i] = a ? sp[i] - other : other - sp[i];
    ds[i] -= (double)nint(ds[i]);
  }
  for (int i = 0; i < 3; ++i) {
    dr[i] = 0.0;
    for (int j = 0; j < 3; ++j) dr[i] += g.h[3 * i + j] * ds[j];
  }
  for (int i = 0; i < 3; ++i) dr2 += dr[i] * dr[i];
  const double length = sqrt(dr2);
  const double stretch = length - g.xr0;
  double tf;
  if (g.xkc >= 0 && stretch < 0)
    tf = g.xkc * stretch;
  else
    tf = g.xk * stretch;
  double F[3];
  for (int i = 0; i < 3; ++i) F[i] = tf * (dr[i] / length);
  double *o = d.xf + 9 * (e >> 1);
  if (a == 0)
    for (int i = 0; i < 3; ++i) o[i] = F[i];
  double dl[3], Fa[3], T[3];
  for (int i = 0; i < 3; ++i) {
    dl[i] = (lam - 0.5 * len) * u[i];
    Fa[i] = a == 0 ? F[i] : -F[i];
  }
  cross3(dl, Fa, T);
  for (int i = 0; i < 3; ++i) o[3 + 3 * a + i] = T[i];
}

// Rebinding: one lane draws for one crosslink; the partner of each that comes
// off is then looked for by 64, 32 or 16 lanes together (for 1, 2 or more in
// the wavefront), a cell of the (2 xreach + 1)^3 neighbourhood a lane.  The
// partner is the candidate of the lowest (score, bond number of the caller),
// whoever finds it.  Few crosslinks come off in a step, so the launch lasts as
// long as one search: 343-729 cells, a chain of loads, roots and divisions for
// each bond in them: 35 us where one lane took 238
// (50k crosslinks, 400k bonds, one coming off).
__global__ __launch_bounds__(kXlBlock) void k_xl_events(Dev d, Geo g) {
  Ctl *ctl = d.ctl;
  if (ctl->abort) return;
  const int64_t x0 = (int64_t)blockIdx.x * kXlBlock;
  const int lane = threadIdx.x;
  const int64_t m = step_index(d) / 2;
  const uint32_t k0 = (uint32_t)g.xseed, k1 = (uint32_t)(g.xseed >> 32);
  uint32_t o[4] = {(uint32_t)(x0 + lane), (uint32_t)((uint64_t)(x0 + lane) >> 32), (uint32_t)m, 1u};
  philox4x32(o, k0, k1);
  uint64_t hits = __ballot(x0 + lane < g.nx && unit_draw(o[0]) < g.xpoff);
  if (!hits) return;
  const int nhit = __popcll(hits);
  const int width = nhit == 1 ? 64 : nhit == 2 ? 32 : 16;  // lanes of a search
  const int n = g.n1d, R = g.xreach;
  const int span = 2 * R + 1 >= n ? n : 2 * R + 1;
  const int off0 = 2 * R + 1 >= n ? 0 : -R;
  while (hits) {
    // the next 64 / width crosslinks, one for each group of lanes
    int src = -1;
    for (int k = 0; k < 64 / width && hits; ++k) {
      const int l = __ffsll((unsigned long long)hits) - 1;
      hits &= hits - 1;
      if (lane / width == k) src = l;
    }
    const uint32_t o1 = __shfl(o[1], src < 0 ? 0 : src), o2 = __shfl(o[2], src < 0 ? 0 : src);
    int32_t best = -1, best_caller = 0;
    uint32_t best_score = 0;
    const int64_t x = x0 + src;
    const int am = unit_draw(o1) < 0.5 ? 0 : 1, as = 1 - am;
    if (src >= 0) {
      const int32_t bs = d.xb[2 * x + as];
      double P[3], u[3], len, sP[3];
      anchor_point(d, g, bs, d.xlam[2 * x + as], P, u, &len);
      scaled(g, P, sP);
      const int32_t key0 = cell_key(n, sP[0], sP[1], sP[2]);
      const int cx = key0 / (n * n), cy = (key0 / n) % n, cz = key0 % n;
      // (cell keys are 32-bit, so the cells of all of the grid are, too)
      for (uint32_t c = lane % width; c < (uint32_t)(span * span * span); c += width) {
        const int dz = (int)(c % span), dy = (int)(c / span % span), dx = (int)(c / span / span);
        const int X = ((cx + off0 + dx) % n + n) % n, Y = ((cy + off0 + dy) % n + n) % n;
        const int Z = ((cz + off0 + dz) % n + n) % n;
        if (!cell_occupied(d, g, X, Y, Z)) continue;  // empty cell
        const int2 run = cell_run_of(d, g, X, Y, Z);
        for (int32_t j = run.x; j < run.y; ++j) {
          const int32_t b = d.sorted[j];
          if (b == bs) continue;
          double rec[7];
          bond_state(d, g, b, rec, rec + 3, rec + 6);
          double ds[3], dr[3], t = 0.0, d2 = 0.0;
          for (int i = 0; i < 3; ++i) {
            ds[i] = rec[i] - sP[i];
            ds[i] -= (double)nint(ds[i]);
          }
          for (int i = 0; i < 3; ++i) {
            dr[i] = 0.0;
            for (int k = 0; k < 3; ++k) dr[i] += g.h[3 * i + k] * ds[k];
          }
          for (int i = 0; i < 3; ++i) t += dr[i] * rec[3 + i];
          const double hl = 0.5 * rec[6];
          if (t > hl) t = hl;
          if (t < -hl) t = -hl;
          for (int i = 0; i < 3; ++i) {
            const double e = dr[i] - t * rec[3 + i];
            d2 += e * e;
          }
          if (!(d2 <= g.xrb2)) continue;
          const int32_t bc = d.bond_caller[b];
          uint32_t q[4] = {(uint32_t)x, (uint32_t)m, (uint32_t)bc, 2u};
          philox4x32(q, k0, k1);
          if (best < 0 || q[0] < best_score || (q[0] == best_score && bc < best_caller)) {
            best = b;
            best_caller = bc;
            best_score = q[0];
          }
        }
      }
    }
    for (int s = width / 2; s > 0; s >>= 1) {
      const int32_t ob = __shfl_xor(best, s), oc = __shfl_xor(best_caller, s);
      const uint32_t os = __shfl_xor(best_score, s);
      if (ob >= 0 && (best < 0 || os < best_score || (os == best_score && oc < best_caller))) {
        best = ob;
        best_caller = oc;
        best_score = os;
      }
    }
    if (best < 0) continue;
    if (lane % width < 9) d.xf[9 * x + lane % width] = 0.0;
    if (lane % width == 0) {
      d.xb[2 * x + am] = best;
      d.xlam[2 * x + am] = unit_draw(o2) * d.fpar[8 * d.bond_fil[best]];
      atomicAdd((unsigned long long *)&ctl->xl_events, 1ull);
      ctl->xl_dirty = 1;
    }
  }
}

// Per-bond lists from the bindings, in one launch: count, chunk sums of the
// counts, starts, fill, sort, with barriers between the passes.  On most steps
// there is no event and the launch returns at once, so what counts is that it
// is one and not six, 1.55 us each.  Blocks for 4096 bonds each, as many as
// the barriers carry.  400k bonds, 50k crosslinks: 84.0 us a step with the six
// launches, 80.0 with this one, which takes 44 us when there was an event.
constexpr int kListBlock = 1024;
constexpr int kXlListBlocks = 128;

__global__ __launch_bounds__(kListBlock) void k_xl_lists(Dev d, Geo g) {
  if (d.ctl->abort || !d.ctl->xl_dirty) return;
  __shared__ int ws[kListBlock / 64];
  int rank, parts;
  if (door_enter(d.door, gridDim.x, &rank, &parts)) {
    const int64_t t0 = (int64_t)rank * kListBlock + threadIdx.x, stride = (int64_t)parts * kListBlock;
    // a block's bonds: a run of whole tiles
    const int64_t tiles = (g.nb + kListBlock - 1) / kListBlock;
    const int64_t b0 = tiles * rank / parts * kListBlock;
    const int64_t b1 = std::min<int64_t>(tiles * (rank + 1) / parts * kListBlock, g.nb);
    for (int64_t e = t0; e < 2 * g.nx; e += stride) atomicAdd(&d.xdeg[d.xb[e]], 1);
    bar_wait(d.door, 0, rank, parts);
    int s = 0;
    for (int64_t b = b0 + threadIdx.x; b < b1; b += kListBlock) s += d.xdeg[b];
    s = block_sum<kListBlock>(s, ws);
    if (threadIdx.x == 0) d.scan_tmp[rank] = s;
    bar_wait(d.door, 1, rank, parts);
    int base = block_sum<kListBlock>((int)threadIdx.x < rank ? d.scan_tmp[threadIdx.x] : 0, ws);
    for (int64_t c = b0; c < b1; c += kListBlock) {
      const int64_t b = c + threadIdx.x;
      int tot;
      const int ex = block_excl<kListBlock>(b < b1 ? d.xdeg[b] : 0, &tot, ws);
      if (b < b1) d.xinc_start[b] = base + ex;
      base += tot;
    }
    if (rank == parts - 1 && threadIdx.x == 0) d.xinc_start[g.nb] = base;
    bar_wait(d.door, 2, rank, parts);
    // places the entries; xdeg returns to zero for the next rebuild
    for (int64_t e = t0; e < 2 * g.nx; e += stride) {
      const int32_t b = d.xb[e];
      d.xinc[d.xinc_start[b] + atomicSub(&d.xdeg[b], 1) - 1] = (int32_t)e;
    }
    bar_wait(d.door, 3, rank, parts);
    for (int64_t b = b0 + threadIdx.x; b < b1; b += kListBlock) {
      const int32_t q0 = d.xinc_start[b], q1 = d.xinc_start[b + 1];
      for (int32_t i = q0 + 1; i < q1; ++i) {
        const int32_t v = d.xinc[i];
        int32_t j = i - 1;
        while (j >= q0 && d.xinc[j] > v) {
          d.xinc[j + 1] = d.xinc[j];
          --j;
        }
        d.xinc[j + 1] = v;
      }
    }
  }
  if (door_leave(d.door, gridDim.x)) {
    if (threadIdx.x == 0) d.ctl->xl_dirty = 0;
    door_reset(d.door);
  }
}

inline dim3 grid_for(int64_t n) {
  const int64_t b = (n + kXlBlock - 1) / kXlBlock;
  return dim3((unsigned)(b > 0 ? b : 1));
}

}  // namespace

void launch_xlink_forces(const Dev &d, const Geo &g, hipStream_t st) {
  if (g.nx <= 0) return;
  hipLaunchKernelGGL(k_xl_force, grid_for(2 * g.nx), dim3(kXlBlock), 0, st, d, g);
}

void launch_xlink_events(const Dev &d, const Geo &g, hipStream_t st) {
  if (g.nx <= 0 || !(g.xpoff > 0)) return;
  hipLaunchKernelGGL(k_xl_events, grid_for(g.nx), dim3(kXlBlock), 0, st, d, g);
}

void launch_xlink_lists(const Dev &d, const Geo &g, hipStream_t st) {
  if (g.nx <= 0) return;
  const int64_t blocks = std::min<int64_t>((g.nb + 4095) / 4096, kXlListBlocks);
  hipLaunchKernelGGL(k_xl_lists, dim3((unsigned)blocks), dim3(kListBlock), 0, st, d, g);
}

}  // namespace sc
