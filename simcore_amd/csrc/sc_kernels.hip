// sc_kernels.hip -- gfx950 kernels of the filament BD step.
//
// Built with -ffp-contract=off: every FP64 multiply and add rounds on its
// own, in the order the reference's source states it, so the FP64 path
// reproduces the CPU path value-for-value.  Division and sqrt on FP64 are
// IEEE correctly rounded on gfx950 (v_div_scale/fmas/fixup sequence and
// the refined v_sqrt_f64 expansion).
//
// One step, in stream order (all guarded by the device control block,
// which holds the decision for the step about to run):
//   [rebuild: keys (+ column populations), column scan, column scatter,
//    column rank sort (+ cell runs, occupancy), degrees, degree sums,
//    incidence lists (+ incidence starts, capacity, zero dr)]
//   -> pair+scatter -> integrate (per length class)
//   -> commit (and decide the next step)
// Runs of odd+even pairs commit less often: an odd step is committed with the
// even step after it, and that pair by the first launch of the next pair
// (fold_commit), so only the last pair of a run needs the commit launch.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sc_block.h"
#include "sc_internal.h"
#include "sc_limits.h"
#include "sc_math.h"

namespace sc {

// ---------------------------------------------------------------------------
// Control kernels
// ---------------------------------------------------------------------------

// Replaces InteractionManager::CheckUpdateInteractions / GetDrMax
// (src/interaction_manager.cpp:284-312) for the step after i_step: the
// accumulator of a full step is compared with 0.25*cell_len^2 at the next
// (odd) step; the mesh skips the update after a midstep
// (src/mesh.cpp:533-536).  A full step clears the accumulator it is about
// to fill.
__device__ __forceinline__ void decide_next(Ctl *c, double thr) {
  const int64_t k = c->i_step + 1;
  c->cur_step = k;
  c->midstep = (k & 1) ? 1 : 0;
  int rb = 0;
  if ((k & 1) && k >= 3) {
    const double drm = __longlong_as_double((long long)c->dr_bits);
    if (drm > 10000) {  // include/simcore/species.hpp:114-118
      c->abort = 1;
      c->err = SC_ERR_UNPHYSICAL;
      return;
    }
    if (drm > thr) rb = 1;
  }
  if (!(k & 1)) c->dr_bits = 0ull;
  c->rebuild = rb;
}

// Folds the per-wave displacement maxima into Ctl::dr_bits and clears the
// slots; one 64-lane block (the launch of k_decide / k_commit).
__device__ __forceinline__ void fold_dr_slots(Ctl *c, unsigned long long *slots) {
  const int lane = threadIdx.x;
  unsigned long long m = 0ull;
  for (int i = lane; i < kDrSlots; i += 64) {
    const unsigned long long v = slots[i];
    m = v > m ? v : m;
    slots[i] = 0ull;
  }
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long y = __shfl_xor(m, o, 64);
    m = y > m ? y : m;
  }
  if (lane == 0 && m > c->dr_bits) c->dr_bits = m;
}

// standalone decision: after loading or after the host changed the state
__global__ void k_decide(Ctl *c, unsigned long long *slots, double thr) {
  if (blockIdx.x != 0 || c->abort) return;
  fold_dr_slots(c, slots);
  if (threadIdx.x == 0) decide_next(c, thr);
}

// end of a step: commit it and decide the next one (one launch for both).
// Every value it needs is loaded up front, so the kernel costs one memory
// round trip; the decision is decide_next's on those values.  `ahead`: the
// odd step before was not committed either (its commit would only have moved
// the counters and cleared dr_bits), so both are committed here.
__device__ __forceinline__ void commit_body(Ctl *c, unsigned long long *slots, double thr,
                                            int ahead) {
  static_assert(kDrSlots == 4 * 64, "four slots per lane");
  const int lane = threadIdx.x;
  unsigned long long v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = slots[lane + 64 * i];
  const int32_t abort = c->abort;
  const int64_t cur = c->cur_step + ahead;
  const unsigned long long drb = ahead ? 0ull : c->dr_bits;
  if (abort) return;
  unsigned long long m = drb;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m = v[i] > m ? v[i] : m;
    slots[lane + 64 * i] = 0ull;
  }
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long y = __shfl_xor(m, o, 64);
    m = y > m ? y : m;
  }
  if (lane != 0) return;
  const int64_t k = cur + 1;  // the next step
  c->i_step = cur;
  c->cur_step = k;
  c->midstep = (k & 1) ? 1 : 0;
  int rb = 0;
  if ((k & 1) && k >= 3) {
    const double drm = __longlong_as_double((long long)m);
    if (drm > 10000) {  // include/simcore/species.hpp:114-118
      c->dr_bits = m;
      c->abort = 1;
      c->err = SC_ERR_UNPHYSICAL;
      return;
    }
    if (drm > thr) rb = 1;
  }
  c->dr_bits = (k & 1) ? m : 0ull;  // a full step clears what it will fill
  c->rebuild = rb;
}

__global__ void k_commit(Ctl *c, unsigned long long *slots, double thr, int ahead) {
  if (blockIdx.x != 0) return;
  commit_body(c, slots, thr, ahead);
}

// one block per member
__global__ void k_group_commit(const Member *__restrict__ ms) {
  const Member &M = ms[blockIdx.x];
  commit_body(M.d[1].ctl, M.d[1].dr_slots, M.g.thr, M.d[1].ahead);
}

__global__ void k_group_ctl(const Member *__restrict__ ms, int n, Ctl *out) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m < n) out[m] = *ms[m].d[0].ctl;
}

__global__ void k_zero_i32(int32_t *p, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) p[i] = 0;
}

__device__ __forceinline__ bool guard_off(const Ctl *c, int guard) {
  if (!c) return false;
  if (c->abort) return true;
  return guard == kGuardRebuild && !c->rebuild;
}

// ---------------------------------------------------------------------------
// Device-wide exclusive scan (int32), three passes.  out has n+1 entries,
// out[n] = total.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int block_excl_scan256(int v, int *total,
                                                  int *wsum) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  int base = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kScanBlock / 64; ++i) {
    int s = wsum[i];
    if (i < w) base += s;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return base + x - v;
}

__device__ __forceinline__ void scan_reduce_body(const int32_t *in, int64_t n, int32_t *bsum,
                                                 int64_t bid, int64_t nblk) {
  __shared__ int wsum[kScanBlock / 64];
  const int64_t ntiles = (n + kScanTile - 1) / kScanTile;
  for (int64_t t = bid; t < ntiles; t += nblk) {
    const int64_t base = t * kScanTile;
    int s = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
      const int64_t i = base + (int64_t)j * kScanBlock + threadIdx.x;
      if (i < n) s += in[i];
    }
    int tot;
    block_excl_scan256(s, &tot, wsum);
    if (threadIdx.x == 0) bsum[t] = tot;
  }
}

__global__ __launch_bounds__(kScanBlock) void k_scan_reduce(
    const int32_t *in, int64_t n, int32_t *bsum, const Ctl *ctl, int guard) {
  if (guard_off(ctl, guard)) return;
  scan_reduce_body(in, n, bsum, blockIdx.x, gridDim.x);
}

__device__ void tile_scan(int *tile, int *wsum, int carry_in, int *total) {
  // tile holds kScanTile ints; exclusive scan in place plus carry_in.
  int v[kScanItems];
  int s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    v[j] = tile[threadIdx.x * kScanItems + j];
    s += v[j];
  }
  int tot;
  int ex = block_excl_scan256(s, &tot, wsum) + carry_in;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    tile[threadIdx.x * kScanItems + j] = ex;
    ex += v[j];
  }
  *total = tot;
  __syncthreads();
}

// Second pass: each tile adds up the sums of the tiles before it (at most a
// few thousand, read from L2) and scans itself; the last tile also writes
// the total.  Two launches per scan; blocks loop over tiles, so any grid
// size serves.
__device__ __forceinline__ void scan_down_body(const int32_t *in, int64_t n, const int32_t *bsum,
                                               int32_t *out, int64_t bid, int64_t nblk) {
  __shared__ int tile[kScanTile];
  __shared__ int wsum[kScanBlock / 64];
  const int64_t ntiles = (n + kScanTile - 1) / kScanTile;
  for (int64_t t = bid; t < ntiles; t += nblk) {
    int part = 0;
    for (int64_t i = threadIdx.x; i < t; i += kScanBlock) part += bsum[i];
    int carry;
    block_excl_scan256(part, &carry, wsum);
    const int64_t base = t * kScanTile;
    for (int j = threadIdx.x; j < kScanTile; j += kScanBlock)
      tile[j] = (base + j < n) ? in[base + j] : 0;
    __syncthreads();
    int tot;
    tile_scan(tile, wsum, carry, &tot);
    for (int j = threadIdx.x; j < kScanTile; j += kScanBlock)
      if (base + j < n) out[base + j] = tile[j];
    if (t == ntiles - 1 && threadIdx.x == 0) out[n] = carry + tot;
    __syncthreads();
  }
}

__global__ __launch_bounds__(kScanBlock) void k_scan_down(const int32_t *in,
                                                          int64_t n,
                                                          const int32_t *bsum,
                                                          int32_t *out,
                                                          const Ctl *ctl,
                                                          int guard) {
  if (guard_off(ctl, guard)) return;
  scan_down_body(in, n, bsum, out, blockIdx.x, gridDim.x);
}

// entries of Dev::scan_tmp: tile sums of a two-launch scan over the columns,
// the degree sums of the list pass, or the crosslink lists' chunk sums
int64_t scan_tmp_elems(int64_t ncol, int64_t nb) {
  const int64_t n = ncol > nb ? ncol : nb;
  const int64_t tiles = (n + kScanTile - 1) / kScanTile + 1;
  const int64_t groups = (nb + kPullGroup - 1) / kPullGroup;
  const int64_t sums = 2 * groups;  // block sums, then group sums
  return tiles > sums ? tiles : sums;
}

void launch_scan(const int32_t *in, int32_t *out, int64_t n, int32_t *tmp,
                 const Ctl *ctl, int guard, hipStream_t st) {
  int64_t nblk = (n + kScanTile - 1) / kScanTile;
  if (nblk == 0) nblk = 1;
  if (nblk > kStreamBlocks) nblk = kStreamBlocks;
  hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)nblk), dim3(kScanBlock), 0,
                     st, in, n, tmp, ctl, guard);
  hipLaunchKernelGGL(k_scan_down, dim3((unsigned)nblk), dim3(kScanBlock), 0,
                     st, in, n, tmp, out, ctl, guard);
}

// ---------------------------------------------------------------------------
// Column starts in one launch.  A tile's block adds up the populations of all
// columns before it itself (at most half a megabyte, in L2, 16 bytes a load)
// instead of waiting for a launch of tile sums: launches cost 1.55 us each
// also on the steps that do not rebuild, and the extra reads take less than
// that up to kColScanMax columns (measured active: 225^2 columns 4.4 us
// against 4.6 + 4.5 for the two launches).  Larger grids of columns keep the
// two-launch scan, whose reads grow linearly.
// ---------------------------------------------------------------------------
constexpr int kColScanBlock = 1024;
constexpr int kColScanTile = 4 * kColScanBlock;
constexpr int64_t kColScanMax = (int64_t)1 << 17;

// (BLOCK threads, a tile of 4 * BLOCK columns)
template <int BLOCK>
__device__ __forceinline__ void colscan_body(const Dev &d, int64_t ncol, int64_t tile) {
  __shared__ int ws[BLOCK / 64];
  const int64_t base = tile * 4 * BLOCK;
  const int4 *in4 = reinterpret_cast<const int4 *>(d.col_count);
  int part = 0;
  for (int64_t i = threadIdx.x; i < base / 4; i += BLOCK) {
    const int4 v = in4[i];
    part += v.x + v.y + v.z + v.w;
  }
  const int carry = block_sum<BLOCK>(part, ws);
  const int64_t i0 = base + 4 * (int64_t)threadIdx.x;
  int v[4], s = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = i0 + k < ncol ? d.col_count[i0 + k] : 0;
    s += v[k];
  }
  int tot;
  int ex = carry + block_excl<BLOCK>(s, &tot, ws);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (i0 + k < ncol) d.col_start[i0 + k] = ex;
    ex += v[k];
  }
  if (base + 4 * BLOCK >= ncol && threadIdx.x == 0) d.col_start[ncol] = carry + tot;
}

__global__ __launch_bounds__(kColScanBlock) void k_colscan(Dev d, int64_t ncol, int guard) {
  if (guard_off(d.ctl, guard)) return;
  colscan_body<kColScanBlock>(d, ncol, blockIdx.x);
}

static inline unsigned colscan_tiles(int64_t ncol) {
  return (unsigned)((ncol + kColScanTile - 1) / kColScanTile);
}

static void launch_colscan(const Dev &d, int64_t ncol, int guard, hipStream_t st) {
  if (ncol <= kColScanMax)
    hipLaunchKernelGGL(k_colscan, dim3(colscan_tiles(ncol)), dim3(kColScanBlock), 0, st, d, ncol,
                       guard);
  else
    launch_scan(d.col_count, d.col_start, ncol, d.scan_tmp, guard ? d.ctl : nullptr, guard, st);
}

// ---------------------------------------------------------------------------
// Rebuild stage
// ---------------------------------------------------------------------------

// CellList::FindCellCoords over every bond (src/cell_list.cpp:139-157) and
// the population of each cell column (x, y) (n1d^2 counters instead of
// n1d^3, so the scan that follows is small), with each bond's place in its
// column.  Streaming passes loop over their range, so any grid size serves.
// The column counts are aggregated per block tile first: each bond enters
// its column into an LDS hash table (linear probing; a tile of BLOCK
// bonds has at most that many columns, so it always fits) and takes its
// place among the tile's bonds of that column from an LDS counter; one
// device-scope atomic per distinct column of the tile then hands out the
// tile's block of places.  With spatially ordered storage a tile touches
// a few tens of columns, so the device-scope atomics (which on MI355X go
// past the XCD's L2 to memory) drop by an order of magnitude.  A bond's
// place is any unique slot of its column; the column sort orders them.
template <int BLOCK>
struct KeysLds {
  int32_t col[BLOCK], cnt[BLOCK], base[BLOCK];
};

template <int BLOCK>
__device__ __forceinline__ void keys_body(const Dev &d, const Geo &g, int64_t bid, int64_t nblk,
                                          KeysLds<BLOCK> &L) {
  int32_t *hcol = L.col, *hcnt = L.cnt, *hbase = L.base;
  constexpr int kHashShift = BLOCK == 1024 ? 22 : BLOCK == 512 ? 23 : 24;  // hash bits: log2(BLOCK)
  static_assert(BLOCK == 256 || BLOCK == 512 || BLOCK == 1024, "hash bits");
  const int t = threadIdx.x;
  const int64_t ntiles = (g.nb + BLOCK - 1) / BLOCK;
  for (int64_t tile = bid; tile < ntiles; tile += nblk) {
    hcol[t] = -1;
    hcnt[t] = 0;
    __syncthreads();
    const int64_t b = tile * BLOCK + t;
    int32_t k = 0, slot = 0, local = 0;
    if (b < g.nb) {
      if (g.compact) {
        k = rec_key_compact(d.br, g, b);
      } else {
        const double *rec = d.br + 8 * b;
        k = cell_key(g.n1d, rec[0], rec[1], rec[2]);
      }
      const int32_t c = k / g.n1d;
      slot = (int32_t)(((uint32_t)c * 2654435761u) >> kHashShift);  // multiplicative hash
      for (;;) {
        const int32_t prev = atomicCAS(&hcol[slot], -1, c);
        if (prev == -1 || prev == c) break;
        slot = (slot + 1) & (BLOCK - 1);
      }
      local = atomicAdd(&hcnt[slot], 1);
    }
    __syncthreads();
    if (hcol[t] >= 0) hbase[t] = atomicAdd(&d.col_count[hcol[t]], hcnt[t]);
    __syncthreads();
    if (b < g.nb) {
      d.keys[b] = k;
      d.col_rank[b] = hbase[slot] + local;
    }
    __syncthreads();
  }
}

// Commit of the full step before an odd step, inside the odd step's first
// launch, in place of a launch of its own (2-3 us, mostly waiting: it is one
// block that loads and stores a few words).  Every block folds the
// displacement slots and takes the decision for itself from values that no
// block of this launch changes; block 0 also stores it in Ctl for the
// launches that follow.  The slots need no clearing for the next full step:
// the accumulators, hence their maximum, only grow until a rebuild zeroes
// them, and the rebuild's column scatter clears the slots too.  Returns
// whether the odd step rebuilds.
__device__ __forceinline__ bool fold_commit(const Dev &d, double thr, bool first) {
  static_assert(kDrSlots == 256, "one slot per thread of the first four wavefronts");
  __shared__ unsigned long long wmax[4];
  __shared__ int off;
  Ctl *c = d.ctl;
  unsigned long long m = threadIdx.x < kDrSlots ? d.dr_slots[threadIdx.x] : 0ull;
  if (threadIdx.x == 0) off = c->abort;
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long y = __shfl_xor(m, o, 64);
    m = y > m ? y : m;
  }
  if ((threadIdx.x & 63) == 0 && threadIdx.x < kDrSlots) wmax[threadIdx.x >> 6] = m;
  __syncthreads();
  if (off) return false;
#pragma unroll
  for (int i = 0; i < 4; ++i) m = wmax[i] > m ? wmax[i] : m;
  const double drm = __longlong_as_double((long long)m);
  const bool lost = drm > 10000;  // include/simcore/species.hpp:114-118
  const bool rb = !lost && drm > thr;
  if (first && threadIdx.x == 0) {
    const int64_t cur = c->cur_step;  // the odd step before the full step
    c->i_step = cur + 1;
    c->cur_step = cur + 2;
    c->dr_bits = m;
    c->rebuild = rb ? 1 : 0;
    if (lost) {
      c->abort = 1;
      c->err = SC_ERR_UNPHYSICAL;
    }
  }
  return rb;
}

template <bool FOLD>
__global__ __launch_bounds__(kScanBlock) void k_keys(Dev d, Geo g) {
  if (FOLD) {
    if (!fold_commit(d, g.thr, blockIdx.x == 0)) return;
  } else {
    if (guard_off(d.ctl, kGuardRebuild)) return;
  }
  __shared__ KeysLds<kScanBlock> L;
  keys_body<kScanBlock>(d, g, blockIdx.x, gridDim.x, L);
}

// Column populations from the stored keys (cell list restore).
__global__ void k_key_count(Dev d, Geo g) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; b < g.nb; b += stride)
    d.col_rank[b] = atomicAdd(&d.col_count[d.keys[b] / g.n1d], 1);
}

// Groups the bonds by column at the place the population count handed
// each bond (order inside a column arbitrary; the rank sort orders it): a
// pure scatter, no atomics.  The key travels with the bond, so the column sort
// need not gather it.
__device__ __forceinline__ void scatter_body(const Dev &d, const Geo &g, int64_t bid,
                                             int64_t nblk) {
  const int64_t stride = nblk * blockDim.x;
  for (int64_t b = bid * blockDim.x + threadIdx.x; b < g.nb; b += stride) {
    const int32_t k = d.keys[b];
    d.col_tmp[d.col_start[k / g.n1d] + d.col_rank[b]] = ((int64_t)k << 32) | (uint32_t)b;
  }
}

// (of the steps before the rebuild, see fold_commit)
__device__ __forceinline__ void clear_dr_slots(const Dev &d) {
  for (int i = threadIdx.x; i < kDrSlots; i += blockDim.x) d.dr_slots[i] = 0ull;
}

__global__ void k_scatter(Dev d, Geo g, int guard) {
  if (guard_off(d.ctl, guard)) return;
  if (blockIdx.x == 0) clear_dr_slots(d);
  scatter_body(d, g, blockIdx.x, gridDim.x);
}

// Each cell column sorted by (cell key, bond index): kColLanes lanes per
// column; an entry's place is the number of smaller (key, bond) pairs in its
// column, counted against the column staged in LDS.  Members of a cell thus
// appear in bond order, the order Cell::AddObj appends in (src/cell.cpp:5-8).
// The pass also writes the column's cell tables: the first sorted entry of
// each occupied cell in z order, at the column's own range of `cell_first`,
// and the column's words of `cell_occ` (every word, so no clearing pass is
// needed), each the occupancy bits of 32 cells and where in `cell_first` the
// first of them stands.  A cell's run is found from its rank among the word's
// bits (cell_run_of) in these small, L2-resident arrays.
//
// A column's lanes lie in one wavefront and share nothing with others, so the
// pass has no block barrier.  Bound: the latency of a column's few loads.
// Sixteen lanes keep 4 columns in flight per wavefront and most lanes busy at
// 2-30 bonds a column.  Active: uneven 1.6M bonds 37 us, dense 620k 18 us (one
// column per wavefront, keys gathered: 7 and 6 us more); in the one-launch rebuild,
// where a few hundred wavefronts serve all columns, 52k bonds gained 1.1 us a
// step.
//
// A wavefront with a column of more than kColStage bonds (large cells, dense
// systems, bundles along z) takes its four one after the other with all 64
// lanes, in all of its LDS: the count is quadratic, and 16 lanes that read the
// column from global memory for each bond took 126 us instead of 24 for 1600
// columns of 90 bonds on average, 560 instead of 77 for 400 of 250, 2530
// instead of 224 for a bundle along z of 256 of 470.
constexpr int kColLanes = 16;
constexpr int kColStage = 96;
constexpr int kColOwn = 4;      // bonds a lane ranks at a time in a long column
constexpr int kOccWords = 44;  // occ_words <= 42 (n1d^3 < 2^31)

template <int BLOCK>
struct ColsortLds {
  int64_t ks[BLOCK / kColLanes][kColStage];  // (key, bond) pairs as they come
  int32_t kr[BLOCK / kColLanes][kColStage];  // the keys in order
  uint32_t occ[BLOCK / kColLanes][kOccWords];
};

// LDS written by lanes of a wavefront is read by its other lanes
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Pairs [from, from + count) of the column at s, padded to whole groups of
// four (which the counts below read together).
template <int LANES>
__device__ __forceinline__ void stage_pairs(const Dev &d, int32_t s, int32_t from, int32_t count,
                                            int lane, int64_t *ks) {
  for (int i = lane; i < ((count + 3) & ~3); i += LANES)
    ks[i] = i < count ? d.col_tmp[s + from + i] : INT64_MAX;
}

// The sort of a column that its LANES lanes hold in LDS.
template <int LANES>
__device__ __forceinline__ void sort_short(const Dev &d, int32_t s, int32_t m, int lane,
                                           int64_t *ks, int32_t *kr) {
  stage_pairs<LANES>(d, s, 0, m, lane, ks);
  wave_sync();
  for (int i = lane; i < m; i += LANES) {
    const int64_t ki = ks[i];
    int32_t r = 0;
    for (int j = 0; j < m; j += 4) {
      const int64_t a = ks[j], b = ks[j + 1], x = ks[j + 2], y = ks[j + 3];
      r += (a < ki) + (b < ki) + (x < ki) + (y < ki);
    }
    kr[r] = (int32_t)(ki >> 32);
    d.sorted[s + r] = (int32_t)(uint32_t)ki;
    d.skey[s + r] = (int32_t)(ki >> 32);
  }
}

// The sort of a column of any length by a wavefront, kColOwn bonds a lane
// against `stage` pairs at a time.
__device__ __forceinline__ void sort_long(const Dev &d, int32_t s, int32_t m, int lane,
                                          int64_t *ks, int32_t *kr, int32_t stage) {
  for (int32_t i0 = 0; i0 < m; i0 += 64 * kColOwn) {
    int64_t own[kColOwn];
    int32_t r[kColOwn];
#pragma unroll
    for (int q = 0; q < kColOwn; ++q) {
      const int32_t i = i0 + 64 * q + lane;
      own[q] = i < m ? d.col_tmp[s + i] : 0;
      r[q] = 0;
    }
    for (int32_t t0 = 0; t0 < m; t0 += stage) {
      const int32_t count = m - t0 < stage ? m - t0 : stage;
      if (i0 == 0 || m > stage) {  // (a column within the stage stays there)
        wave_sync();
        stage_pairs<64>(d, s, t0, count, lane, ks);
        wave_sync();
      }
      for (int j = 0; j < count; j += 4) {
        const int64_t a = ks[j], b = ks[j + 1], x = ks[j + 2], y = ks[j + 3];
#pragma unroll
        for (int q = 0; q < kColOwn; ++q)
          r[q] += (a < own[q]) + (b < own[q]) + (x < own[q]) + (y < own[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < kColOwn; ++q)
      if (i0 + 64 * q + lane < m) {
        if (m <= stage) kr[r[q]] = (int32_t)(own[q] >> 32);
        d.sorted[s + r[q]] = (int32_t)(uint32_t)own[q];
        d.skey[s + r[q]] = (int32_t)(own[q] >> 32);
      }
  }
  // (read back below from global memory when not in LDS)
  if (m > stage) __threadfence();
}

// The cell tables of column c, bonds [s, s + m) of the sorted order; each run
// start's rank among the column's run starts comes from a ballot per LANES
// entries.  `held`: the sorted keys are in kr; `rounds` the same for all lanes
// of the wavefront; `shift` the lanes' place in a ballot.
template <int LANES>
__device__ __forceinline__ void column_tables(const Dev &d, const Geo &g, int64_t c, bool live,
                                              int32_t s, int32_t m, bool held, int rounds,
                                              int lane, int shift, const int32_t *kr,
                                              uint32_t *occ) {
  const int n = g.n1d, W = g.occ_words;
  const int64_t ncol = (int64_t)n * n;
  const int32_t e = s + m;
  int32_t ncell = 0;
  for (int q = 0; q < rounds; ++q) {
    const int i = q * LANES + lane;
    int32_t k = -1;
    bool start = false;
    if (i < m) {
      k = held ? kr[i] : d.skey[s + i];
      const int32_t kp = i == 0 ? -1 : (held ? kr[i - 1] : d.skey[s + i - 1]);
      start = k != kp;
    }
    unsigned long long bal = __ballot(start) >> shift;
    if (LANES < 64) bal &= (1ull << (LANES & 63)) - 1;
    if (start) {
      const int32_t rank = ncell + __popcll(bal & ((1ull << lane) - 1ull));
      d.cell_first[s + rank] = s + i;
      const int p = k - (int32_t)c * n + 1;
      atomicOr(&occ[p >> 5], 1u << (p & 31));
    }
    ncell += __popcll(bal);
  }
  wave_sync();
  if (!live) return;
  // (the copies of the first and the last cell beyond the ends count for no
  // run index)
  const uint32_t below = (occ[n >> 5] >> (n & 31)) & 1u, above = (occ[0] >> 1) & 1u;
  for (int w = lane; w < W; w += LANES) {
    int at = s;
    for (int v = 0; v < w; ++v) at += __popc(occ[v]);
    uint32_t bits = occ[w];
    if (w == 0) {
      bits |= below;
      at -= (int)below;
    }
    if (w == (n + 1) >> 5) bits |= above << ((n + 1) & 31);
    d.cell_occ[c * W + w] = make_int2((int32_t)bits, at);
  }
  // where the last run of the column ends (the first of the next column
  // starts there if every bond is a run of its own)
  if (lane == 0 && ncell < m) d.cell_first[s + ncell] = e;
  if (lane == 0 && c == ncol - 1) d.cell_first[e] = e;
}

template <int BLOCK>
__device__ __forceinline__ void colsort_body(const Dev &d, const Geo &g, int64_t bid,
                                             int64_t nblk, ColsortLds<BLOCK> &L) {
  constexpr int kCols = BLOCK / kColLanes, kWaveCols = 64 / kColLanes;
  const int col = threadIdx.x / kColLanes, lane = threadIdx.x % kColLanes;
  const int wlane = threadIdx.x & 63, col0 = col / kWaveCols * kWaveCols;
  const int W = g.occ_words;
  const int64_t ncol = (int64_t)g.n1d * g.n1d;
  const int64_t ngrp = (ncol + kCols - 1) / kCols;
  for (int64_t grp = bid; grp < ngrp; grp += nblk) {
    const int64_t c = grp * kCols + col;
    const bool live = c < ncol;
    const int32_t s = live ? d.col_start[c] : 0, m = live ? d.col_start[c + 1] - s : 0;
    for (int w = lane; w < W; w += kColLanes) L.occ[col][w] = 0u;
    if (live && lane == 0) d.col_count[c] = 0;  // for the next build's count
    int longest = m;
    for (int o = kColLanes; o < 64; o <<= 1) {
      const int y = __shfl_xor(longest, o, 64);
      longest = y > longest ? y : longest;
    }
    if (longest <= kColStage) {
      sort_short<kColLanes>(d, s, m, lane, L.ks[col], L.kr[col]);
      wave_sync();
      // (the wavefront's columns take the longest one's rounds)
      column_tables<kColLanes>(d, g, c, live, s, m, true, (longest + kColLanes - 1) / kColLanes,
                               lane, wlane - lane, L.kr[col], L.occ[col]);
    } else {
      for (int k = 0; k < kWaveCols; ++k) {
        const int64_t ck = grp * kCols + col0 + k;
        const int32_t sk = __shfl(s, k * kColLanes, 64), mk = __shfl(m, k * kColLanes, 64);
        wave_sync();
        // (the four columns' stages are one piece of memory)
        int32_t *kr = &L.kr[0][0] + col0 * kColStage;
        sort_long(d, sk, mk, wlane, &L.ks[0][0] + col0 * kColStage, kr, kWaveCols * kColStage);
        wave_sync();
        column_tables<64>(d, g, ck, ck < ncol, sk, mk, mk <= kWaveCols * kColStage, (mk + 63) / 64,
                          wlane, 0, kr, L.occ[col0 + k]);
      }
    }
    wave_sync();
  }
}

constexpr int kColBlock = 256;
constexpr int64_t kColBlocks = 1024;  // (blocks loop over the columns)

__global__ __launch_bounds__(kColBlock) void k_colsort(Dev d, Geo g, int guard) {
  if (guard_off(d.ctl, guard)) return;
  __shared__ ColsortLds<kColBlock> L;
  colsort_body<kColBlock>(d, g, blockIdx.x, gridDim.x, L);
}

static inline unsigned colsort_grid(int64_t ncol) {
  constexpr int kCols = kColBlock / kColLanes;
  return (unsigned)std::min<int64_t>((ncol + kCols - 1) / kCols, kColBlocks);
}

// The 27 cells around (x, y, z) are numbered (dx + 1) + 3 (dy + 1) +
// 9 (dz + 1): 13 is the cell itself, 14 + q the q-th cell of its half shell in
// the order of CellList::AssignCellNeighbors (src/cell_list.cpp:206-262):
// (x+1, y, z); (x-1..x+1, y+1, z); then (x-1..x+1, y-1..y+1, z+1), x fastest;
// and 12 - q the q-th cell of the mirrored half shell, the 13 cells whose half
// shell holds (x, y, z).  Periodic wrap; with at least 3 cells per side the 27
// are distinct.
constexpr int kOwnCell = 13;

__device__ __forceinline__ void stencil_cell(int n, int x, int y, int z, int code, int *xo, int *yo,
                                             int *zo) {
  const int xp = x + code % 3 - 1, yp = y + code / 3 % 3 - 1, zp = z + code / 9 - 1;
  *xo = xp < 0 ? n - 1 : (xp == n ? 0 : xp);
  *yo = yp < 0 ? n - 1 : (yp == n ? 0 : yp);
  *zo = zp < 0 ? n - 1 : (zp == n ? 0 : zp);
}

// Occupancy of the 27 cells around (and with) cell (cx, cy, cz).  Nine independent loads, one for each column: two words
// of its table hold the bits of cz - 1, cz and cz + 1, also across the
// periodic faces.  (26 loads, one a cell, and three more for each run kept the
// load units of k_deg 70% busy.  Active, 1.6M uneven bonds: k_deg 114 ->
// 103 us, k_colsort 44 -> 37 without its table of runs by cell.)
__device__ __forceinline__ uint32_t stencil_mask(const Dev &d, const Geo &g, int cx, int cy,
                                                 int cz) {
  const int n = g.n1d;
  const int xs[3] = {cx == 0 ? n - 1 : cx - 1, cx, cx == n - 1 ? 0 : cx + 1};
  const int ys[3] = {cy == 0 ? n - 1 : cy - 1, cy, cy == n - 1 ? 0 : cy + 1};
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const int64_t c = (int64_t)xs[i % 3] * n + ys[i / 3];
    int4 w;  // {bits, index} of two words
    __builtin_memcpy(&w, d.cell_occ + c * g.occ_words + (cz >> 5), sizeof(w));
    const uint64_t bits = (uint32_t)w.x | (uint64_t)(uint32_t)w.z << 32;
    const uint32_t v = (uint32_t)(bits >> (cz & 31));
    m |= ((v & 1u) << i) | (((v >> 1) & 1u) << (9 + i)) | (((v >> 2) & 1u) << (18 + i));
  }
  return m;
}

// Geo::home_order of a cell
__device__ __forceinline__ uint64_t home_order_of(const Geo &g, int cx, int cy, int cz) {
  const int n = g.n1d;
  return g.home_order[(cx == 0 ? 0 : cx == n - 1 ? 2 : 1) * 6 +
                      (cy == 0 ? 0 : cy == n - 1 ? 2 : 1) * 2 + (cz == 0 ? 0 : 1)];
}

// The bonds b-1 and b+1 when they share a site with b (Bond::HasNeighbor
// within one mesh, src/bond.cpp:118-121): the pairs the reference culls on
// the rebuild step (src/interaction_manager.cpp:485-497), never listed here.
struct Excl {
  int32_t lo, hi;  // b-1 / b+1, or -1
};

__device__ __forceinline__ Excl excl_of(const Dev &d, const Geo &g, int32_t b) {
  const int32_t f = d.bond_fil[b];
  Excl x;
  x.lo = (b > 0 && d.bond_fil[b - 1] == f) ? b - 1 : -1;
  x.hi = (b + 1 < g.nb && d.bond_fil[b + 1] == f) ? b + 1 : -1;
  return x;
}

// Degree of every bond: the candidates that list it (Cell::MakePairs,
// src/cell.cpp:14-70): the other members of its cell, the members of its 13
// half-shell cells and of its 13 mirrored half-shell cells, less the
// site-sharing neighbours among them.  One thread per sorted position (the
// cell lookups of neighbouring threads then hit the same lines; in bond order
// the pass took 133 us instead of 103 at 1.6M uneven bonds), no atomics.
//
// The runs go to the bond's slab in the order of its list, so the list pass,
// which runs in bond order, only copies them: kSlabRuns starts, as many
// lengths of a byte, and a word {runs | place of the own cell's run << 8 |
// half-shell runs << 16}, 64 bytes, one whole line (the scattered stores waste
// nothing).  Bonds with more runs (a mean of 4.5-5.2, at most 16 seen) or a
// longer one are marked kSlabOver, and the list pass looks theirs up.
constexpr int kSlabRuns = 12;
constexpr int32_t kSlabOver = INT32_MIN;

__device__ __forceinline__ void deg_one(const Dev &d, const Geo &g, int64_t p) {
  const int32_t k = d.skey[p];
  const int32_t b = d.sorted[p];
  const Excl x = excl_of(d, g, b);
  const int32_t klo = x.lo >= 0 ? d.keys[x.lo] : -1;
  const int32_t khi = x.hi >= 0 ? d.keys[x.hi] : -1;
  const int n = g.n1d;
  const int cx = k / (n * n), cy = (k / n) % n, cz = k % n;
  const uint32_t m = stencil_mask(d, g, cx, cy, cz);
  // the occupied cells in list order, 5 bits each
  uint64_t seq = 0, order = home_order_of(g, cx, cy, cz);
  int runs = 0, own_at = 0;
  auto add = [&](int code) {
    if (runs < kSlabRuns) seq |= (uint64_t)code << (5 * runs);
    ++runs;
  };
  for (int step = 0; step < 14; ++step, order >>= 4) {
    const int c = (int)(order & 15);
    if (c == 13) {
      own_at = runs;
      add(kOwnCell);
      for (uint32_t h = m >> 14; h; h &= h - 1) add(13 + __ffs(h));
    } else if ((m >> (12 - c)) & 1u) {
      add(12 - c);
    }
  }
  int32_t start[kSlabRuns], deg = -1;
  uint32_t len[kSlabRuns];
  bool over = runs > kSlabRuns;
  auto run_of = [&](int code) {  // counts the run, too
    int x, y, z;
    stencil_cell(n, cx, cy, cz, code, &x, &y, &z);
    const int2 r = cell_run_of(d, g, x, y, z);
    const int32_t kc = (x * n + y) * n + z;
    deg += (r.y - r.x) - (klo == kc) - (khi == kc);
    return r;
  };
#pragma unroll
  for (int i = 0; i < kSlabRuns; ++i) {
    start[i] = 0;
    len[i] = 0;
    if (i < runs) {
      const int2 r = run_of((int)(seq >> (5 * i)) & 31);
      start[i] = r.x;
      len[i] = (uint32_t)(r.y - r.x);
      over = over || r.y - r.x > 255;
    }
  }
  if (runs > kSlabRuns) {  // all of them again
    deg = -1;
    for (uint32_t h = m; h; h &= h - 1) run_of(__ffs(h) - 1);
  }
  d.deg[b] = deg;
  int4 *slab = reinterpret_cast<int4 *>(d.slab + (int64_t)b * kSlabWords);
  static_assert(kSlabWords == 16 && kSlabRuns == 12, "four int4 stores per slab");
  slab[0] = make_int4(start[0], start[1], start[2], start[3]);
  slab[1] = make_int4(start[4], start[5], start[6], start[7]);
  slab[2] = make_int4(start[8], start[9], start[10], start[11]);
  auto four = [&](int i) {
    return (int32_t)(len[i] | len[i + 1] << 8 | len[i + 2] << 16 | len[i + 3] << 24);
  };
  slab[3] = make_int4(four(0), four(4), four(8),
                      over ? kSlabOver : runs | own_at << 8 | __popc(m >> 14) << 16);
}

// Grid-stride over the sorted positions: a capped grid keeps the launch
// cheap on the steps that do not rebuild (the guard returns at once).
__device__ __forceinline__ void deg_body(const Dev &d, const Geo &g, int64_t bid, int64_t nblk) {
  const int64_t stride = nblk * blockDim.x;
  for (int64_t p = bid * blockDim.x + threadIdx.x; p < g.nb; p += stride) deg_one(d, g, p);
}

__global__ __launch_bounds__(256) void k_deg(Dev d, Geo g) {
  if (guard_off(d.ctl, kGuardRebuild)) return;
  deg_body(d, g, blockIdx.x, gridDim.x);
}

// Degree sums of the groups of kPullGroup bonds and of blocks of kSuper such
// groups, one 256-thread block per kSuper groups.  The list pass scans its own
// group and adds up the blocks and groups before it, so the degrees need no
// scan of their own (one launch instead of two, and the incidence starts are
// written by the pass that uses them).  With group sums alone every block of
// the list pass read all of them, which cost the uneven 1.6M-bond system 1 us
// per step more than the two-launch scan; two levels read one block sum per
// thread there.  A wavefront sums one group: with eight of them one after the
// other (32 groups a block) the launch took 11.2 us instead of 5.1, 620k bonds
// 78.8 -> 78.3 us a step.  Layout in Dev::scan_tmp: the block sums, then the
// group sums.
constexpr int kSuper = 4;

__device__ __forceinline__ int64_t n_groups(int64_t nb) { return (nb + kPullGroup - 1) / kPullGroup; }
__device__ __forceinline__ int64_t n_supers(int64_t nb) {
  return (nb + kPullGroup * kSuper - 1) / (kPullGroup * kSuper);
}

__device__ __forceinline__ void degsum_body(const Dev &d, const Geo &g, int64_t sup) {
  __shared__ int64_t ws[4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int32_t *gsum = d.scan_tmp + n_supers(g.nb);
  const int64_t ngrp = n_groups(g.nb);
  static_assert(kSuper == 4, "a group per wavefront");
  const int64_t grp = sup * kSuper + wv;
  int64_t all = 0;
#pragma unroll
  for (int k = 0; k < kPullGroup / 64; ++k) {
    const int64_t b = grp * kPullGroup + lane + 64 * k;
    if (b < g.nb) all += d.deg[b];
  }
  for (int o = 32; o > 0; o >>= 1) all += __shfl_xor(all, o, 64);
  if (lane == 0 && grp < ngrp) gsum[grp] = kept_length(all);
  if (lane == 0) ws[wv] = all;
  __syncthreads();
  if (threadIdx.x == 0) d.scan_tmp[sup] = kept_length(ws[0] + ws[1] + ws[2] + ws[3]);
}

__global__ __launch_bounds__(256) void k_degsum(Dev d, Geo g) {
  if (guard_off(d.ctl, kGuardRebuild)) return;
  degsum_body(d, g, blockIdx.x);
}

static inline unsigned degsum_blocks(int64_t nb) {
  return (unsigned)std::max<int64_t>(1, (nb + kPullGroup * kSuper - 1) / (kPullGroup * kSuper));
}

// Incidence lists in candidate order, one thread per bond, no atomics and
// no sort.  The list order of CellList::MakePairs (src/cell_list.cpp:
// 127-137, src/cell.cpp:14-70) is: home cells in key order; inside a home
// cell its self pairs (i < j, in member order), then for each of its 13
// half-shell cells in stencil order all (home member, neighbour member)
// pairs, home member outer.  So bond b's candidates come from its own cell
// (as obj2 of the self pairs with earlier members, as obj1 of those with
// later members, then as obj1 of its rows of the 13 half-shell blocks) and
// from each occupied mirrored half-shell cell m (as obj2 of m's block
// toward b's cell, one pair per member of m, in member order), the groups
// taken in home-key order.  That order of the 14 home cells depends only on
// which of b's cell coordinates sit on a periodic face (Geo::home_order,
// built on the host), so no per-thread sort is needed.  Entries {partner,
// role | written << 1 | (b mod 64) << 2}: the owner's place in its 64-bond
// group lets the balanced pair kernel find an entry's bond without a
// search; the slot copies start unwritten (zero force).  The launch also
// checks the capacity, commits the list length and restarts the
// displacement bookkeeping (InteractionManager::ZeroDrTot -> Mesh/Object::
// ZeroDrTot, src/interaction_manager.cpp:316-321, src/mesh.cpp:546-551).
// k_deg leaves the runs in that order, so the pass copies them with their
// first members loaded ahead.  When it walked the stencil itself, each cell a
// branch and a load that waited, it was half the time on vector instructions
// and half on loads, active: uneven 1.6M bonds 139 us, dense 620k 56; now 108
// and 38, and k_deg 4 more.  Eight wavefronts a SIMD: 124 and 39 with the six
// that 74 registers allow.
// Where a failed list pass reports to: Ctl's own words, or, while blocks of
// the same launch may still read those, words that reach Ctl at its end.
struct Failure {
  int32_t *abort, *err, *overflow;
};

__device__ __forceinline__ Failure ctl_failure(const Dev &d) {
  return {&d.ctl->abort, &d.ctl->err, &d.ctl->overflow};
}

__device__ __forceinline__ void pull_one(const Dev &d, const Geo &g, int32_t b,
                                         int32_t w, int32_t wend, int2 *stage,
                                         int32_t base, const Failure &fail) {
  const Excl x = excl_of(d, g, b);
  const int32_t tag = (b & 63) << 2;
  auto put = [&](int32_t a, int role) {
    if (a == b || a == x.lo || a == x.hi) return;
    if (w < wend) {
      if (stage)
        stage[w - base] = make_int2(a, role | tag);
      else
        d.inc[w] = make_int2(a, role | tag);
    }
    ++w;
  };
  const int4 *sl = reinterpret_cast<const int4 *>(d.slab + (int64_t)b * kSlabWords);
  const int4 s0 = sl[0], s1 = sl[1], s2 = sl[2], s3 = sl[3];
  if (s3.w != kSlabOver) {
    const int32_t start[kSlabRuns] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y,
                                      s1.z, s1.w, s2.x, s2.y, s2.z, s2.w};
    const uint32_t len[3] = {(uint32_t)s3.x, (uint32_t)s3.y, (uint32_t)s3.z};
    const int runs = s3.w & 255, own = (s3.w >> 8) & 255, half = s3.w >> 16;
    // the first member of every run (mostly its only one), in flight together
    int32_t first[kSlabRuns];
#pragma unroll
    for (int i = 0; i < kSlabRuns; ++i)
      if (i < runs) first[i] = d.sorted[start[i]];
#pragma unroll
    for (int i = 0; i < kSlabRuns; ++i) {
      if (i < runs) {
        // own cell: obj2 of the pairs with earlier members, obj1 of those
        // with later ones; half shell: obj1; mirrored half shell: obj2
        const int32_t pivot = i == own ? b : i > own && i <= own + half ? INT32_MIN : INT32_MAX;
        put(first[i], first[i] < pivot);
        const int l = (int)((len[i / 4] >> (8 * (i % 4))) & 255u);
        for (int j = 1; j < l; ++j) {
          const int32_t a = d.sorted[start[i] + j];
          put(a, a < pivot);
        }
      }
    }
  } else {
    const int32_t k = d.keys[b];
    const int n = g.n1d;
    const int cx = k / (n * n), cy = (k / n) % n, cz = k % n;
    const uint32_t m = stencil_mask(d, g, cx, cy, cz);
    auto walk = [&](int code, int32_t pivot) {
      int x, y, z;
      stencil_cell(n, cx, cy, cz, code, &x, &y, &z);
      const int2 r = cell_run_of(d, g, x, y, z);
      for (int32_t j = r.x; j < r.y; ++j) {
        const int32_t a = d.sorted[j];
        put(a, a < pivot);
      }
    };
    uint64_t order = home_order_of(g, cx, cy, cz);
    for (int step = 0; step < 14; ++step, order >>= 4) {
      const int c = (int)(order & 15);
      if (c == 13) {
        walk(kOwnCell, b);
        for (uint32_t h = m >> 14; h; h &= h - 1) walk(13 + __ffs(h), INT32_MIN);
      } else if ((m >> (12 - c)) & 1u) {
        walk(12 - c, INT32_MAX);
      }
    }
  }
  if (w != wend) {  // degree and list disagree: never expected; fail the step
    *fail.abort = 1;
    *fail.err = SC_ERR_STATE;
  }
}

constexpr int kPullStage = 512;

// Each 256 threads of a block take every so-many-th group of kPullGroup
// bonds; the list range of a group starts at the sum of the groups before it.
// The total is 64-bit and its parts are cut off rather than wrapped
// (kept_length), so a count that does not fit the lists is seen before
// anything is written.
template <int BLOCK>
struct PullLds {
  int64_t red[BLOCK / 64];
  int2 stage[BLOCK / 64][kPullStage];
  int ws[BLOCK / 64];
};

template <int BLOCK, bool SUMS>
__device__ __forceinline__ void pull_body(const Dev &d, const Geo &g, int64_t bid, int64_t nblk,
                                          const Failure &fail, PullLds<BLOCK> &L) {
  static_assert(kPullGroup == 256, "one bond per thread");
  constexpr int kSubs = BLOCK / 256;
  int64_t *red = L.red;
  int *ws = L.ws;
  const int t = threadIdx.x % 256, sub = threadIdx.x / 256, wv = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t i0 = bid * BLOCK + threadIdx.x;
  const int64_t stride = nblk * BLOCK;
  const int64_t ngrp = n_groups(g.nb), nsup = n_supers(g.nb);
  int64_t part = 0;
  int32_t before = 0;  // (of no use unless the total fits)
  if (SUMS) {
    for (int64_t i = threadIdx.x; i < nsup; i += BLOCK) part += d.scan_tmp[i];
  } else {
    const int4 *deg4 = reinterpret_cast<const int4 *>(d.deg);
    const int64_t first = bid * BLOCK / 4, n4 = g.nb / 4;
    for (int64_t i = threadIdx.x; i < n4; i += BLOCK) {
      const int4 v = deg4[i];
      const int64_t four = (int64_t)v.x + v.y + v.z + v.w;
      part += four;
      if (i < first) before += (int32_t)four;
    }
    // (the last one to three bonds come before no block's first)
    if (4 * n4 + threadIdx.x < g.nb) part += d.deg[4 * n4 + threadIdx.x];
  }
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
  if (lane == 0) red[wv] = part;
  __syncthreads();
  int64_t total = 0;  // two per candidate
#pragma unroll
  for (int i = 0; i < BLOCK / 64; ++i) total += red[i];
  const bool fits = total <= 2 * g.cap;
  if (i0 == 0) {
    d.ctl->nc_need = candidates_of(total);
    if (fits) {
      d.ctl->nc = total / 2;
      d.ctl->n_rebuilds += 1;
      d.inc_start[g.nb] = (int32_t)total;
    } else {
      *fail.abort = 1;
      *fail.overflow = 1;
    }
  }
  if (!fits) return;
  for (int64_t i = i0; i < g.ns; i += stride) {
    for (int q = 0; q < 3; ++q) d.dr0[q * g.ns + i] = d.r[q * g.ns + i];
    d.acc[i] = 0.0;
  }
  // the incidence starts of the block's groups, before the walk over them (in
  // one loop with it they cost the walk 22 registers, two waves per SIMD)
  if (SUMS) {
    static_assert(!SUMS || BLOCK == 256, "a group per block");
    for (int grp = (int)bid; grp < (int)ngrp; grp += (int)nblk) {
      const int64_t b = (int64_t)grp * kPullGroup + t;
      const int sup = grp / kSuper;
      int32_t ahead = sup * kSuper + t < grp ? d.scan_tmp[nsup + sup * kSuper + t] : 0;
      for (int i = t; i < sup; i += 256) ahead += d.scan_tmp[i];
      const int32_t base = block_sum<256>(ahead, ws);
      int gtot;
      const int32_t w = base + block_excl<256>(b < g.nb ? d.deg[b] : 0, &gtot, ws);
      if (b < g.nb) d.inc_start[b] = w;  // read back by the same thread below
    }
  } else {
    int32_t base = block_sum<BLOCK>(before, ws);
    for (int64_t b0 = bid * BLOCK; b0 < g.nb; b0 += stride) {
      const int64_t b = b0 + threadIdx.x;
      int tot;
      const int32_t w = base + block_excl<BLOCK>(b < g.nb ? d.deg[b] : 0, &tot, ws);
      if (b < g.nb) d.inc_start[b] = w;
      // (to the block's next bonds, if there are any)
      int32_t skip = 0;
      if (b0 + stride < g.nb)
        for (int64_t i = b + BLOCK; i < b0 + stride; i += BLOCK) skip += d.deg[i];
      base += tot + block_sum<BLOCK>(skip, ws);
    }
  }
  // each wavefront's 64 consecutive bonds have one contiguous list range:
  // written to LDS entry by entry, then copied out in coalesced stores
  // (ranges longer than the stage are written directly)
  for (int64_t grp0 = bid * kSubs; grp0 < ngrp; grp0 += nblk * kSubs) {
    const int64_t b = (grp0 + sub) * kPullGroup + t;
    int32_t w = (int32_t)total, wend = w;
    if (b < g.nb) {
      w = d.inc_start[b];
      wend = w + d.deg[b];
    }
    const int32_t base = __shfl(w, 0, 64), cnt = __shfl(wend, 63, 64) - base;
    const bool staged = cnt <= kPullStage;
    if (b < g.nb) pull_one(d, g, (int32_t)b, w, wend, staged ? L.stage[wv] : nullptr, base, fail);
    wave_sync();
    if (staged)
      for (int i = lane; i < cnt; i += 64) d.inc[base + i] = L.stage[wv][i];
    wave_sync();
  }
}

__global__ __launch_bounds__(256, 8) void k_pull(Dev d, Geo g) {
  if (guard_off(d.ctl, kGuardRebuild)) return;
  __shared__ PullLds<256> L;
  pull_body<256, true>(d, g, blockIdx.x, gridDim.x, ctl_failure(d), L);
}

// ---- the rebuild stage in one launch ----------------------------------------
// Every launch costs 1.55 us also on a step that does not rebuild, so one
// launch runs the passes where it can, with a barrier between them among its
// blocks (sc_block.h): 3.5 us among 64 blocks, 7 among 256, against 1.55 us for
// a kernel boundary; hence few, large blocks.  The seven launches serve what
// wants more of them.  us a step, seven launches against one:
//   many bonds (up to 256k every thread of 256 blocks has one bond): 1k 25.7 /
//     22.4, FP64 1.2k 31.4 / 27.3, 52k 31.9 / 29.6, 62k with stress sums 34.2 /
//     31.6, 155k 41.6 / 39.4, FP64 155k 55.4 / 53.6, FP64 uneven 230k 92.4 /
//     89.0, 232k 47.5 / 47.3, 372k 60.9 / 66.4;
//   many columns, whose sort is the longest pass (a rebuild every eleventh
//     step): 200^2 with 300 bonds 22.6 / 20.7, with 5000 25.3 / 24.6, 256^2
//     23.0 / 22.3 and 25.5 / 26.2, 362^2 24.0 / 26.5 and 26.8 / 31.6;
//   long lists, whose gathers want every CU (the same): 64k bonds with 30
//     entries each 97.6 / 98.7, with 127 381 / 387, 150k with 18 139.5 / 141.4;
//     16k (in blocks of 512) with 57 115.3 / 112.8, with 130 237.7 / 236.2.
//
// The list pass adds up the degrees itself: with few bonds that is less than
// the pass of group sums and its barrier, 11 us of a rebuild of 85 at 52k
// bonds (27.5 -> 27.1 us a step, 62k with stress sums 29.2 -> 28.9).
constexpr int64_t kOneLaunchBonds = 262144;
constexpr int64_t kOneLaunchColumns = (int64_t)1 << 16;

// Threads of a block: the gathers of the degree and list passes keep a CU's
// load units busy, so small systems spread their bonds over more CUs with
// blocks of 512 until the barriers cost more.  512 against 1024, us a step: 1k
// bonds 18.2 / 18.6, 10k 20.1 / 20.5, 31k 23.2 / 23.5, 62k 28.0 / 27.5, 102k
// 34.3 / 32.7.
constexpr int64_t kSmallBonds = 40960;

// (the lists have to get a quarter shorter again before one launch is back)
bool rebuild_in_one(const Geo &g, double mean, bool now) {
  const double line = (g.nb <= kSmallBonds ? 160.0 : 16.0) * (now ? 1.0 : 0.75);
  return g.nb <= kOneLaunchBonds && (int64_t)g.n1d * g.n1d <= kOneLaunchColumns && mean <= line;
}

// Blocks of the one launch: enough for 800 bonds each (64 or 128 blocks were
// the best of 16 to 256 at 52k and 101k bonds; at 155k 1200 bonds a block cost
// 1.5 us a step more), 400 in blocks of 512, and in small sparse systems for
// 64 columns each, whose sort is the longest pass there.
static inline unsigned one_blocks(const Geo &g, int block) {
  const int64_t ncol = (int64_t)g.n1d * g.n1d, per = block == 512 ? 400 : 800;
  const int64_t b = std::max<int64_t>((g.nb + per - 1) / per, std::min<int64_t>((ncol + 63) / 64, 64));
  return (unsigned)std::min<int64_t>(std::max<int64_t>(b, 1), 256);
}

// Blocks of a batch up to which its members rebuild in one launch.  The chip
// holds 256 of 1024 threads or 512 of 512 at once: with more, also a step on
// which nobody rebuilds takes a round of blocks after the other (about 3 us
// each), and members wait for blocks that find no room.  us a step of the
// batch, seven launches / one, and the one's blocks: 16 x 10k bonds 87.5 / 79.6
// with 576, 8 x 31k 88.5 / 85.4 with 624, 8 x 50k 102.9 / 95.7 with 496, 12 x
// 50k 118.8 / 115.8 with 744, 8 x 40k 98.1 / 100.2 with 808, 24 x 50k 175 / 194
// with 1488, 8 x 87k 126 / 156 with 872, 16 x 87k 193 / 285 with 1744.
constexpr int32_t kBatchBlocks = 768;

// The block that leaves last: until then a block that comes late must still
// find the rebuild decided as the others did, or it would leave uncounted; so
// what the decision is taken from -- the displacement slots, Ctl's abort word
// -- changes only here.
__device__ __forceinline__ void rebuild_one_end(const Dev &d) {
  clear_dr_slots(d);
  if (threadIdx.x != 0) return;
  Door *b = d.door;
  Ctl *c = d.ctl;
  if (b->overflow) c->overflow = 1;
  if (b->err) c->err = b->err;
  if (b->abort) c->abort = 1;
  b->overflow = b->err = b->abort = 0;
}

// the passes' stages, one after the other in the same memory
template <int BLOCK>
union OneLds {
  KeysLds<BLOCK> keys;
  ColsortLds<BLOCK> col;
  PullLds<BLOCK> pull;
};

template <int BLOCK, bool FOLD>
__device__ __forceinline__ void rebuild_one_body(const Dev &d, const Geo &g, uint32_t blocks,
                                                 bool first, OneLds<BLOCK> &L) {
  if (FOLD) {
    if (!fold_commit(d, g.thr, first)) return;
  } else {
    if (guard_off(d.ctl, kGuardRebuild)) return;
  }
  Door *door = d.door;
  int rank, parts;
  if (door_enter(door, blocks, &rank, &parts)) {
    const int64_t ncol = (int64_t)g.n1d * g.n1d;
    keys_body<BLOCK>(d, g, rank, parts, L.keys);
    bar_wait(door, 0, rank, parts);
    for (int64_t t = rank; t * 4 * BLOCK < ncol; t += parts)
      colscan_body<BLOCK>(d, ncol, t);
    bar_wait(door, 1, rank, parts);
    scatter_body(d, g, rank, parts);
    bar_wait(door, 2, rank, parts);
    colsort_body<BLOCK>(d, g, rank, parts, L.col);
    bar_wait(door, 3, rank, parts);
    deg_body(d, g, rank, parts);
    bar_wait(door, 4, rank, parts);
    const Failure fail = {&door->abort, &door->err, &door->overflow};
    pull_body<BLOCK, false>(d, g, rank, parts, fail, L.pull);
  }
  if (door_leave(door, blocks)) {
    rebuild_one_end(d);
    door_reset(door);
  }
}

template <int BLOCK, bool FOLD>
__global__ __launch_bounds__(BLOCK) void k_rebuild_one(Dev d, Geo g) {
  __shared__ OneLds<BLOCK> L;
  rebuild_one_body<BLOCK, FOLD>(d, g, gridDim.x, blockIdx.x == 0, L);
}

static inline unsigned nblocks(int64_t n, int bs) {
  int64_t b = (n + bs - 1) / bs;
  return (unsigned)(b > 0 ? b : 1);
}

static inline unsigned sgrid(int64_t n) {
  const unsigned b = nblocks(n, 256);
  return b < (unsigned)kStreamBlocks ? b : (unsigned)kStreamBlocks;
}

// One launch (k_rebuild_one) where rebuild_in_one says so; else
// keys (+ column populations) -> column scan -> column scatter -> column
// sort (+ runs, occupancy) -> degrees -> degree sums -> incidence lists
// (+ incidence starts, capacity check, displacement restart): 7 launches,
// none over the n1d^3 cells.  Every launch's grid is capped (the kernels
// loop over their range), so on the odd steps that do not rebuild each
// launch only reads the guard.  The two per-bond list passes are
// latency-bound and get 8 waves per SIMD.
constexpr unsigned kListBlocks = 2048;

void launch_rebuild(const Dev &d, const Geo &g, bool fold, hipStream_t st) {
  const unsigned gs = sgrid(g.nb);
  const int64_t ncol = (int64_t)g.n1d * g.n1d;
  if (g.one_launch) {
    const dim3 grid(one_blocks(g, g.nb <= kSmallBonds ? 512 : 1024));
    if (g.nb <= kSmallBonds && fold)
      hipLaunchKernelGGL((k_rebuild_one<512, true>), grid, dim3(512), 0, st, d, g);
    else if (g.nb <= kSmallBonds)
      hipLaunchKernelGGL((k_rebuild_one<512, false>), grid, dim3(512), 0, st, d, g);
    else if (fold)
      hipLaunchKernelGGL((k_rebuild_one<1024, true>), grid, dim3(1024), 0, st, d, g);
    else
      hipLaunchKernelGGL((k_rebuild_one<1024, false>), grid, dim3(1024), 0, st, d, g);
    return;
  }
  if (fold)
    hipLaunchKernelGGL(k_keys<true>, dim3(gs), dim3(kScanBlock), 0, st, d, g);
  else
    hipLaunchKernelGGL(k_keys<false>, dim3(gs), dim3(kScanBlock), 0, st, d, g);
  launch_colscan(d, ncol, kGuardRebuild, st);
  hipLaunchKernelGGL(k_scatter, dim3(gs), dim3(kScanBlock), 0, st, d, g, (int)kGuardRebuild);
  hipLaunchKernelGGL(k_colsort, dim3(colsort_grid(ncol)), dim3(kColBlock), 0, st, d, g,
                     (int)kGuardRebuild);
  const unsigned gl = std::min(nblocks(g.nb, 256), kListBlocks);
  hipLaunchKernelGGL(k_deg, dim3(gl), dim3(256), 0, st, d, g);
  hipLaunchKernelGGL(k_degsum, dim3(degsum_blocks(g.nb)), dim3(256), 0, st, d, g);
  hipLaunchKernelGGL(k_pull, dim3(std::min(nblocks(g.ns > g.nb ? g.ns : g.nb, 256), kListBlocks)),
                     dim3(256), 0, st, d, g);
}

// Ensemble batches: the launches of launch_rebuild, each over all members
// (odd-step pointers: a rebuild only ever starts an odd step); a member
// that does not rebuild returns at its guard.  Threads of a block and bonds of
// a wavefront follow from the whole batch, so a member's grid need not be that
// of its own launch; no kernel's results depend on its grid.
template <bool FOLD>
__global__ __launch_bounds__(kScanBlock) void k_group_keys(const Member *__restrict__ ms,
                                                           GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  if (FOLD) {
    if (!fold_commit(M.d[0], M.g.thr, (int)blockIdx.x == b0)) return;
  } else {
    if (guard_off(M.d[0].ctl, kGuardRebuild)) return;
  }
  __shared__ KeysLds<kScanBlock> L;
  keys_body<kScanBlock>(M.d[0], M.g, blockIdx.x - b0, nblk, L);
}

__global__ void k_group_scatter(const Member *__restrict__ ms, GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  if (guard_off(M.d[0].ctl, kGuardRebuild)) return;
  if ((int)blockIdx.x == b0) clear_dr_slots(M.d[0]);
  scatter_body(M.d[0], M.g, blockIdx.x - b0, nblk);
}

__global__ __launch_bounds__(kColBlock) void k_group_colsort(const Member *__restrict__ ms,
                                                             GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  if (guard_off(M.d[0].ctl, kGuardRebuild)) return;
  __shared__ ColsortLds<kColBlock> L;
  colsort_body<kColBlock>(M.d[0], M.g, blockIdx.x - b0, nblk, L);
}

__global__ __launch_bounds__(256) void k_group_deg(const Member *__restrict__ ms, GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  if (guard_off(M.d[0].ctl, kGuardRebuild)) return;
  deg_body(M.d[0], M.g, blockIdx.x - b0, nblk);
}

__global__ __launch_bounds__(256) void k_group_pull(const Member *__restrict__ ms, GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  if (guard_off(M.d[0].ctl, kGuardRebuild)) return;
  __shared__ PullLds<256> L;
  pull_body<256, true>(M.d[0], M.g, blockIdx.x - b0, nblk, ctl_failure(M.d[0]), L);
}

// the two-launch column scan, for batches with a member of more than
// kColScanMax columns
__global__ __launch_bounds__(kScanBlock) void k_group_scan_reduce(const Member *__restrict__ ms,
                                                                  GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  const Dev &d = M.d[0];
  if (guard_off(d.ctl, kGuardRebuild)) return;
  scan_reduce_body(d.col_count, (int64_t)M.g.n1d * M.g.n1d, d.scan_tmp, blockIdx.x - b0, nblk);
}

__global__ __launch_bounds__(kScanBlock) void k_group_scan_down(const Member *__restrict__ ms,
                                                                GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  const Dev &d = M.d[0];
  if (guard_off(d.ctl, kGuardRebuild)) return;
  scan_down_body(d.col_count, (int64_t)M.g.n1d * M.g.n1d, d.scan_tmp, d.col_start,
                 blockIdx.x - b0, nblk);
}

__global__ __launch_bounds__(kColScanBlock) void k_group_colscan(const Member *__restrict__ ms,
                                                                 GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  if (guard_off(M.d[0].ctl, kGuardRebuild)) return;
  colscan_body<kColScanBlock>(M.d[0], (int64_t)M.g.n1d * M.g.n1d, blockIdx.x - b0);
}

__global__ __launch_bounds__(256) void k_group_degsum(const Member *__restrict__ ms,
                                                      GroupGrid gg) {
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  if (guard_off(M.d[0].ctl, kGuardRebuild)) return;
  degsum_body(M.d[0], M.g, blockIdx.x - b0);
}

template <int BLOCK, bool FOLD>
__global__ __launch_bounds__(BLOCK) void k_group_rebuild_one(const Member *__restrict__ ms,
                                                                 GroupGrid gg) {
  __shared__ OneLds<BLOCK> L;
  int b0, nblk;
  const Member &M = ms[group_member(gg, blockIdx.x, &b0, &nblk)];
  rebuild_one_body<BLOCK, FOLD>(M.d[0], M.g, nblk, (int)blockIdx.x == b0, L);
}

namespace {
// offsets of a grouped launch from each member's block count; the total
template <typename F>
int32_t group_grid(GroupGrid &gg, const Member *hm, int n, F blocks) {
  int32_t t = 0;
  for (int m = 0; m < n; ++m) {
    gg.off[m] = t;
    t += (int32_t)blocks(hm[m].g);
  }
  for (int m = n; m <= kMaxGroup; ++m) gg.off[m] = t;
  return t;
}

unsigned scan_blocks(int64_t n) {
  const int64_t nblk = std::max<int64_t>(1, (n + kScanTile - 1) / kScanTile);
  return (unsigned)std::min<int64_t>(nblk, kStreamBlocks);
}
}  // namespace

void launch_group_rebuild(const Member *dm, const Member *hm, int n, bool fold, hipStream_t st) {
  if (n <= 0) return;
  bool one = true;
  bool small = true;
  for (int m = 0; m < n; ++m) {
    one = one && hm[m].g.one_launch;
    small = small && hm[m].g.nb <= kSmallBonds;
  }
  GroupGrid go;
  const int32_t to = group_grid(go, hm, n, [small](const Geo &g) {
    return one_blocks(g, small ? 512 : 1024);
  });
  if (one && to <= kBatchBlocks) {
    if (small && fold)
      hipLaunchKernelGGL((k_group_rebuild_one<512, true>), dim3(to), dim3(512), 0, st, dm, go);
    else if (small)
      hipLaunchKernelGGL((k_group_rebuild_one<512, false>), dim3(to), dim3(512), 0, st, dm, go);
    else if (fold)
      hipLaunchKernelGGL((k_group_rebuild_one<1024, true>), dim3(to), dim3(1024), 0, st, dm, go);
    else
      hipLaunchKernelGGL((k_group_rebuild_one<1024, false>), dim3(to), dim3(1024), 0, st, dm, go);
    return;
  }
  GroupGrid gk, gcs, gsrt, gdeg, gds, gpl;
  const int32_t tk = group_grid(gk, hm, n, [](const Geo &g) { return sgrid(g.nb); });
  bool wide = false;
  for (int m = 0; m < n; ++m) wide = wide || (int64_t)hm[m].g.n1d * hm[m].g.n1d > kColScanMax;
  const int32_t tcs = group_grid(gcs, hm, n, [wide](const Geo &g) {
    const int64_t ncol = (int64_t)g.n1d * g.n1d;
    return wide ? scan_blocks(ncol) : colscan_tiles(ncol);
  });
  const int32_t tsrt = group_grid(gsrt, hm, n, [](const Geo &g) {
    return colsort_grid((int64_t)g.n1d * g.n1d);
  });
  const int32_t tdeg = group_grid(gdeg, hm, n, [](const Geo &g) {
    return std::min(nblocks(g.nb, 256), kListBlocks);
  });
  const int32_t tds = group_grid(gds, hm, n, [](const Geo &g) { return degsum_blocks(g.nb); });
  const int32_t tpl = group_grid(gpl, hm, n, [](const Geo &g) {
    return std::min(nblocks(g.ns > g.nb ? g.ns : g.nb, 256), kListBlocks);
  });
  if (fold)
    hipLaunchKernelGGL(k_group_keys<true>, dim3(tk), dim3(kScanBlock), 0, st, dm, gk);
  else
    hipLaunchKernelGGL(k_group_keys<false>, dim3(tk), dim3(kScanBlock), 0, st, dm, gk);
  if (wide) {
    hipLaunchKernelGGL(k_group_scan_reduce, dim3(tcs), dim3(kScanBlock), 0, st, dm, gcs);
    hipLaunchKernelGGL(k_group_scan_down, dim3(tcs), dim3(kScanBlock), 0, st, dm, gcs);
  } else {
    hipLaunchKernelGGL(k_group_colscan, dim3(tcs), dim3(kColScanBlock), 0, st, dm, gcs);
  }
  hipLaunchKernelGGL(k_group_scatter, dim3(tk), dim3(kScanBlock), 0, st, dm, gk);
  hipLaunchKernelGGL(k_group_colsort, dim3(tsrt), dim3(kColBlock), 0, st, dm, gsrt);
  hipLaunchKernelGGL(k_group_deg, dim3(tdeg), dim3(256), 0, st, dm, gdeg);
  hipLaunchKernelGGL(k_group_degsum, dim3(tds), dim3(256), 0, st, dm, gds);
  hipLaunchKernelGGL(k_group_pull, dim3(tpl), dim3(256), 0, st, dm, gpl);
}

void launch_group_commit(const Member *dm, int n, hipStream_t st) {
  if (n > 0) hipLaunchKernelGGL(k_group_commit, dim3(n), dim3(64), 0, st, dm);
}

void launch_group_ctl(const Member *dm, int n, Ctl *out, hipStream_t st) {
  if (n > 0) hipLaunchKernelGGL(k_group_ctl, dim3(1), dim3(64), 0, st, dm, n, out);
}

// The cell list of the last rebuild (sorted, runs, occupancy) from the
// stored keys; after a checkpoint restore the crosslink partner search
// needs the list the saved state was stepping with.
void launch_cells_from_keys(const Dev &d, const Geo &g, hipStream_t st) {
  const int64_t ncol = (int64_t)g.n1d * g.n1d;
  hipLaunchKernelGGL(k_key_count, dim3(sgrid(g.nb)), dim3(256), 0, st, d, g);
  launch_colscan(d, ncol, 0, st);
  hipLaunchKernelGGL(k_scatter, dim3(sgrid(g.nb)), dim3(256), 0, st, d, g, 0);
  hipLaunchKernelGGL(k_colsort, dim3(colsort_grid(ncol)), dim3(kColBlock), 0, st, d, g, 0);
}

// Replays the displacement bookkeeping of the last full step after the host
// replaced the site positions: acc = acc_prev + 2 |r - r0|^2 with the new
// positions, the order Object::UpdateDrTot adds in (src/object.cpp:282-287).
__global__ void k_redo_dr(Dev d, Geo g) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double a = 0.0;
  if (i < g.ns) {
    a = d.acc_prev[i];
    for (int rep = 0; rep < 2; ++rep)
      for (int k = 0; k < 3; ++k) {
        double dd = d.r[k * g.ns + i] - d.dr0[k * g.ns + i];
        a += dd * dd;
      }
    d.acc[i] = a;
  }
  for (int o = 32; o > 0; o >>= 1) {
    double y = __shfl_xor(a, o, 64);
    a = y > a ? y : a;
  }
  if ((threadIdx.x & 63) == 0)
    atomicMax(&d.dr_slots[(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) &
                          (kDrSlots - 1)],
              (unsigned long long)__double_as_longlong(a));
}

void launch_redo_dr(const Dev &d, const Geo &g, hipStream_t st) {
  hipLaunchKernelGGL(k_redo_dr, dim3(nblocks(g.ns, 256)), dim3(256), 0, st, d, g);
}

// Plain streaming copy, the calibration kernel for HBM byte counters.
__global__ void k_copy_probe(const double4 *__restrict__ src, double4 *__restrict__ dst,
                             int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += st) dst[i] = src[i];
}

void launch_copy_probe(const void *src, void *dst, int64_t n32, hipStream_t st) {
  hipLaunchKernelGGL(k_copy_probe, dim3(4096), dim3(256), 0, st, (const double4 *)src,
                     (double4 *)dst, n32);
}

void launch_decide(const Dev &d, const Geo &g, hipStream_t st) {
  hipLaunchKernelGGL(k_decide, dim3(1), dim3(64), 0, st, d.ctl, d.dr_slots, g.thr);
}

void launch_commit(const Dev &d, const Geo &g, hipStream_t st) {
  hipLaunchKernelGGL(k_commit, dim3(1), dim3(64), 0, st, d.ctl, d.dr_slots, g.thr, d.ahead);
}

void launch_zero_i32(int32_t *p, int64_t n, hipStream_t st) {
  unsigned gb = nblocks(n, 256);
  if (gb > 4096) gb = 4096;
  hipLaunchKernelGGL(k_zero_i32, dim3(gb), dim3(256), 0, st, p, n);
}

__global__ void k_bond_init(Dev d, Geo g, int prec) {
  int f = blockIdx.x * blockDim.y + threadIdx.y;
  if (f >= g.nf) return;
  const int64_t s0 = d.site_off[f], s1 = d.site_off[f + 1];
  const int64_t b0 = s0 - f;
  for (int64_t i = threadIdx.x; i < s1 - s0 - 1; i += blockDim.x) {
    double r1[3], r2[3];
    for (int k = 0; k < 3; ++k) {
      r1[k] = d.r[k * g.ns + s0 + i];
      r2[k] = d.r[k * g.ns + s0 + i + 1];
    }
    bond_reinit(d, g, b0 + i, r1, r2, prec);
  }
}

void launch_bond_init(const Dev &d, const Geo &g, int precision,
                      hipStream_t st) {
  dim3 bs(64, 4);
  hipLaunchKernelGGL(k_bond_init, dim3(nblocks(g.nf, 4)), bs, 0, st, d, g,
                     precision);
}

}  // namespace sc
