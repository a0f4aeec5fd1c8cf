// sc_analysis.hip -- on-device filament analyses: end-to-end vectors,
// centres of mass (FilamentSpecies::RunMse2eAnalysis,
// src/filament_species.cpp:569-593) and the cos(theta) histogram of
// consecutive bonds (RunThetaAnalysis, :595-610).  Read-only over the state;
// cheap next to a step, so long statistical runs can sample often.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sc_internal.h"
#include "sc_math.h"

namespace sc {

namespace {

// Lanes per filament of the statistics and caller-order passes: a segment's
// loads fill whole 128-byte lines, and a filament of the usual 8-64 sites
// keeps most of its lanes busy.
constexpr int kFilLanes = 16;

// kFilLanes lanes per filament: its sites are read in coalesced runs and the
// centre of mass summed by a lane tree (one thread per filament read strided
// 8-byte elements: 16.9 us on the dense 620k-bond system).  Results go to the
// caller's filament order, so the host only copies them out.  Bound: latency
// of one pass over the positions.
__global__ __launch_bounds__(256) void k_filament_stats(Dev d, Geo g, double *e2e,
                                                        double *com) {
  const int f = blockIdx.x * (256 / kFilLanes) + (int)threadIdx.x / kFilLanes;
  const int gl = threadIdx.x % kFilLanes;
  if (f >= g.nf) return;  // whole groups leave together
  const int64_t s0 = d.site_off[f], s1 = d.site_off[f + 1];
  const int64_t ns = g.ns, nf = g.nf;
  const int u = d.fil_caller[f];
  for (int q = 0; q < 3; ++q) {
    const double *r = d.r + q * ns;
    if (e2e && gl == 0) e2e[q * nf + u] = r[s1 - 1] - r[s0];
    if (com) {
      double s = 0.0;
      for (int64_t i = s0 + gl; i < s1; i += kFilLanes) s += r[i];
#pragma unroll
      for (int o = kFilLanes / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, kFilLanes);
      if (gl == 0) com[q * nf + u] = s / (double)(s1 - s0);
    }
  }
}

// Histogram cell of bond j and its successor: angle index (j - first bond of
// the filament) and cos = u_j . u_{j+1}; -1 when j is a filament's last bond
// or its row is past n_rows.
__device__ __forceinline__ int64_t theta_cell(const Dev &d, const Geo &g, int64_t j, int n_bins,
                                              int n_rows) {
  const int f = d.bond_fil[j];
  const int64_t b0 = d.site_off[f] - f;
  const int64_t b1 = d.site_off[f + 1] - f - 1;  // one past the last bond
  if (j + 1 >= b1) return -1;
  const int row = (int)(j - b0);
  if (row >= n_rows) return -1;
  double s[3], a[3], b[3], l;
  rec_read(d.br, g, j, s, a, &l);
  rec_read(d.br, g, j + 1, s, b, &l);
  const double c = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
  int bin = (int)floor((1.0 + c) * (n_bins / 2));
  if (bin >= n_bins) bin = n_bins - 1;
  if (bin < 0) bin = 0;
  return (int64_t)row * n_bins + bin;
}

// One thread per bond, one device-scope atomic per count: for shapes beyond
// the LDS of k_theta_hist_lds.
__global__ __launch_bounds__(256) void k_theta_hist(Dev d, Geo g, int n_bins, int n_rows,
                                                    unsigned long long *hist) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= g.nb) return;
  const int64_t c = theta_cell(d, g, j, n_bins, n_rows);
  if (c >= 0) atomicAdd(&hist[c], 1ull);
}

// Counts of a block's bonds in LDS, added to the result once per block and
// non-empty cell.  Stiff filaments put nearly every count of a row into its
// last few bins, and device-scope atomics on one address serialise (about
// 25 ns each), so the per-bond form took 183 us for 620k bonds, 31 rows.  At
// most 512 blocks: the adds per address stay few.
constexpr int kThetaLds = 8192;  // counters: 32 KB, five blocks per CU
constexpr int kThetaBlocks = 512;

__global__ __launch_bounds__(256) void k_theta_hist_lds(Dev d, Geo g, int n_bins, int n_rows,
                                                        unsigned long long *hist) {
  extern __shared__ uint32_t cnt[];
  const int n = n_bins * n_rows;
  for (int i = threadIdx.x; i < n; i += 256) cnt[i] = 0u;
  __syncthreads();
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < g.nb; j += stride) {
    const int64_t c = theta_cell(d, g, j, n_bins, n_rows);
    if (c >= 0) atomicAdd(&cnt[c], 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 256)
    if (cnt[i]) atomicAdd(&hist[i], (unsigned long long)cnt[i]);
}

// Storage-order array (n entries per component, sites or bonds of every
// filament) to the caller's order in FP64: kFilLanes lanes per filament, both
// sides in coalesced runs.  Bound: one read and one write of the array.
template <typename T>
__global__ __launch_bounds__(256) void k_caller_order(Dev d, Geo g, const T *__restrict__ src,
                                                      double *__restrict__ dst, int64_t n,
                                                      int comp, int bonds) {
  const int f = blockIdx.x * (256 / kFilLanes) + (int)threadIdx.x / kFilLanes;
  const int gl = threadIdx.x % kFilLanes;
  if (f >= g.nf) return;
  const int64_t s0 = d.site_off[f] - (bonds ? f : 0);
  const int64_t len = d.site_off[f + 1] - d.site_off[f] - bonds;
  const int64_t t0 = d.noise_off[f] - (bonds ? d.fil_caller[f] : 0);
  for (int k = 0; k < comp; ++k)
    for (int64_t i = gl; i < len; i += kFilLanes) dst[k * n + t0 + i] = (double)src[k * n + s0 + i];
}

inline dim3 fil_grid(int nf) {
  const int per = 256 / kFilLanes, b = (nf + per - 1) / per;
  return dim3((unsigned)(b > 0 ? b : 1));
}

}  // namespace

void launch_filament_stats(const Dev &d, const Geo &g, double *e2e, double *com,
                           hipStream_t st) {
  hipLaunchKernelGGL(k_filament_stats, fil_grid(g.nf), dim3(256), 0, st, d, g, e2e, com);
}

void launch_theta_hist(const Dev &d, const Geo &g, int n_bins, int n_rows,
                       unsigned long long *hist, hipStream_t st) {
  const int64_t blocks = std::max<int64_t>(1, (g.nb + 255) / 256);
  const int64_t n = (int64_t)n_bins * n_rows;
  if (n <= kThetaLds)
    hipLaunchKernelGGL(k_theta_hist_lds, dim3((unsigned)std::min<int64_t>(blocks, kThetaBlocks)),
                       dim3(256), (size_t)n * sizeof(uint32_t), st, d, g, n_bins, n_rows, hist);
  else
    hipLaunchKernelGGL(k_theta_hist, dim3((unsigned)blocks), dim3(256), 0, st, d, g, n_bins,
                       n_rows, hist);
}

void launch_caller_order(const Dev &d, const Geo &g, const void *src, bool f32, double *dst,
                         int64_t n, int comp, bool bonds, hipStream_t st) {
  if (f32)
    hipLaunchKernelGGL(k_caller_order<float>, fil_grid(g.nf), dim3(256), 0, st, d, g,
                       static_cast<const float *>(src), dst, n, comp, bonds ? 1 : 0);
  else
    hipLaunchKernelGGL(k_caller_order<double>, fil_grid(g.nf), dim3(256), 0, st, d, g,
                       static_cast<const double *>(src), dst, n, comp, bonds ? 1 : 0);
}

}  // namespace sc
