// sdpd_cells.hip -- K1: cell list by a stable counting sort (gfx950).
//
// Replaces technique_build_list -> ppm_neighlist_clist -> ppm_util_rank3d
// (ppm.tgz:src/ppm_util_rank3d.F90:395-531).  The reference sorts particle
// indices into boxes with a stable counting sort: histogram, prefix sum,
// scatter in ascending particle index.  Here:
//   1. key + histogram   one thread per particle; the cell key is PPM's
//                        FLOOR((x - x0) * rdx) with its upper-face
//                        corrections; the slot inside the cell comes from an
//                        integer atomic (arrival order, not yet stable)
//   2. scan              exclusive prefix sum of the cell counts
//   3. scatter           unsorted[start[key] + slot] = i
//   4. place             each particle ranks itself among the members of its
//                        cell by index (the stable order the reference
//                        produces), then moves its state to that slot
// The result is identical run to run and equal to the reference's
// lhbx / lpdx for the same particle order.  Particles stay in cell order
// between steps, so the next sort is a near-identity permutation and the
// place pass writes almost coalesced.
#include <algorithm>

#include "sdpd_kernels.h"

namespace sdpd {

__global__ void k_fill_i32(int32_t* __restrict__ a, int32_t v, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) a[i] = v;
}

__global__ void k_fill_f64(double* __restrict__ a, double v, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) a[i] = v;
}

// Exclusive scan of count[0..m) into start[0..m] in three passes over
// tiles of 4096 entries: tile sums, a scan of the tile sums in one
// workgroup, and the tile scans with their offsets.
constexpr int kScanTile = 4096;

__device__ __forceinline__ int32_t block_exclusive_scan_1024(int32_t v, int32_t& total,
                                                             int32_t* wsum) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  int32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    int32_t t = __shfl_up(incl, off, 64);
    if (lane >= off) incl += t;
  }
  if (lane == 63) wsum[wid] = incl;
  __syncthreads();
  if (wid == 0) {
    int32_t s = lane < 16 ? wsum[lane] : 0;
    int32_t si = s;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      int32_t t = __shfl_up(si, off, 64);
      if (lane >= off) si += t;
    }
    if (lane < 16) wsum[lane] = si - s;
    if (lane == 15) wsum[16] = si;
  }
  __syncthreads();
  total = wsum[16];
  int32_t r = wsum[wid] + incl - v;
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(1024) void k_scan_tile_sums(const int32_t* __restrict__ count,
                                                         int32_t* __restrict__ sums, int32_t m) {
  __shared__ int32_t wsum[17];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x * 4;
  int32_t local = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (base + q < m) local += count[base + q];
  int32_t total;
  (void)block_exclusive_scan_1024(local, total, wsum);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(1024) void k_scan_sums(int32_t* __restrict__ sums, int32_t ntile,
                                                    int32_t* __restrict__ out_total) {
  __shared__ int32_t wsum[17];
  __shared__ int32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int32_t b0 = 0; b0 < ntile; b0 += 1024) {
    const int32_t idx = b0 + threadIdx.x;
    const int32_t v = idx < ntile ? sums[idx] : 0;
    int32_t total;
    const int32_t ex = block_exclusive_scan_1024(v, total, wsum);
    const int32_t c = carry;
    if (idx < ntile) sums[idx] = c + ex;
    __syncthreads();
    if (threadIdx.x == 0) carry = c + total;
    __syncthreads();
  }
  if (threadIdx.x == 0) *out_total = carry;
}

__global__ __launch_bounds__(1024) void k_scan_tiles(const int32_t* __restrict__ count,
                                                     const int32_t* __restrict__ sums,
                                                     int32_t* __restrict__ start, int32_t m) {
  __shared__ int32_t wsum[17];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x * 4;
  int32_t v[4], local = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    v[q] = base + q < m ? count[base + q] : 0;
    local += v[q];
  }
  int32_t total;
  int32_t ex = block_exclusive_scan_1024(local, total, wsum) + sums[blockIdx.x];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (base + q < m) start[base + q] = ex;
    ex += v[q];
  }
}

// start[m] receives the total
static void launch_exclusive_scan(hipStream_t s, const int32_t* count, int32_t* start, int32_t m,
                                  int32_t* tile_sums) {
  const int32_t ntile = (m + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL(k_scan_tile_sums, dim3(ntile), dim3(1024), 0, s, count, tile_sums, m);
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(1024), 0, s, tile_sums, ntile, start + m);
  hipLaunchKernelGGL(k_scan_tiles, dim3(ntile), dim3(1024), 0, s, count, tile_sums, start, m);
}

__global__ void k_scatter(int n, const int32_t* __restrict__ key, const int32_t* __restrict__ slot,
                          const int32_t* __restrict__ start, int32_t* __restrict__ unsorted) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  unsorted[start[key[i]] + slot[i]] = i;
}

// ---------------------------------------------------------------------
// the sort of the step, as items of work in phases
// ---------------------------------------------------------------------
// Phases (each needs all of the one before):
//   keys     cell key, slot and histogram       1024 particles per item
//   sums     sums of 4096 cell counts           one tile per item
//   starts   first particle of every cell       one tile per item, which adds
//                                               up the sums of the tiles before
//   scatter  unsorted[start[key] + slot] = i    1024 particles; item 0 is the
//                                               pair kernels' work map
//   place    rank in the cell, state moved to the *_alt buffers, cell counts
//            cleared for the next sort          1024 particles
//   back     the state copied back, with x_ref and the walks' positions
//                                               1024 particles (Verlet lists)
// The counts are zero between sorts.
constexpr int kSortThreads = 256;
constexpr int kSortItem = 1024;
enum SortPhase { kKeys = 0, kSums, kStarts, kScatter, kPlace, kBack, kSortPhases };

struct SortPlan {
  int32_t items[kSortPhases];
  int32_t copy_back;
};

static SortPlan sort_plan(const DevParams& P, bool keys, bool copy_back) {
  const int32_t blocks = (P.n + kSortItem - 1) / kSortItem;
  const int32_t tiles = (P.ncell + kScanTile - 1) / kScanTile;
  return {{keys ? blocks : 0, tiles, tiles, blocks + 1, blocks, copy_back ? blocks : 0},
          copy_back ? 1 : 0};
}

// exclusive scan over the workgroup's 256 threads
__device__ __forceinline__ int32_t block_scan_256(int32_t v, int32_t& total, int32_t* wsum) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t t = __shfl_up(incl, off, 64);
    if (lane >= off) incl += t;
  }
  if (lane == 63) wsum[wid] = incl;
  __syncthreads();
  const int32_t a = wsum[0], b = wsum[1], c = wsum[2], d = wsum[3];
  total = a + b + c + d;
  const int32_t before = wid == 0 ? 0 : (wid == 1 ? a : (wid == 2 ? a + b : a + b + c));
  __syncthreads();
  return before + incl - v;
}

__device__ __forceinline__ void sort_keys(const DevParams& P, const DeviceState& S, int item) {
  const int64_t n = P.n;
  for (int q = 0; q < kSortItem / kSortThreads; ++q) {
    const int i0 = item * kSortItem + q * kSortThreads + (int)threadIdx.x;
    const bool act = i0 < P.n;
    const int i = act ? i0 : P.n - 1;  // every lane takes part in the histogram
    const RepGeom& g = S.geo[S.rep[i]];
    const int32_t k =
        cell_key_geo(g, P.dim, S.x[i], S.x[n + i], P.dim == 3 ? S.x[2 * n + i] : 0.0);
    const int32_t sl = histogram_slot(S.count, k, act);
    if (act) {
      S.key[i] = k;
      S.slot[i] = sl;
    }
  }
}

__device__ __forceinline__ void sort_sums(const DevParams& P, const DeviceState& S, int item,
                                          int32_t* wsum) {
  const int64_t base = (int64_t)item * kScanTile + threadIdx.x * (kScanTile / kSortThreads);
  int32_t local = 0;
  for (int q = 0; q < kScanTile / kSortThreads; ++q)
    if (base + q < P.ncell) local += S.count[base + q];
  int32_t total;
  (void)block_scan_256(local, total, wsum);
  if (threadIdx.x == 0) S.scan_tmp[item] = total;
}

__device__ __forceinline__ void sort_starts(const DevParams& P, const DeviceState& S, int item,
                                            int32_t* wsum) {
  int32_t part = 0, before;
  for (int t = threadIdx.x; t < item; t += kSortThreads) part += S.scan_tmp[t];
  (void)block_scan_256(part, before, wsum);
  constexpr int kPer = kScanTile / kSortThreads;
  const int64_t base = (int64_t)item * kScanTile + threadIdx.x * kPer;
  int32_t v[kPer], local = 0;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    v[q] = base + q < P.ncell ? S.count[base + q] : 0;
    local += v[q];
  }
  int32_t total;
  int32_t ex = block_scan_256(local, total, wsum) + before;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    if (base + q < P.ncell) S.start[base + q] = ex;
    ex += v[q];
  }
  if (threadIdx.x == 0 && (int64_t)(item + 1) * kScanTile >= P.ncell) S.start[P.ncell] = before + total;
}

// Work map of the pair kernels: each (y, z) row of the sort grid is cut
// into chunks of at most 64 consecutive particles; chunk c belongs to row
// chunk_row[c] and is the (c - row_chunk_off[row])-th chunk of that row.
__device__ __forceinline__ void sort_rows(const DevParams& P, const DeviceState& S,
                                          int32_t* wsum) {
  constexpr int kPer = 4;
  int32_t carry = 0;
  for (int r0 = 0; r0 < P.nrows; r0 += kPer * kSortThreads) {
    const int base = r0 + (int)threadIdx.x * kPer;
    int32_t nc[kPer], local = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      nc[q] = 0;
      if (base + q < P.nrows) {
        const int c0 = S.row_cell[base + q];
        nc[q] = (S.start[c0 + S.row_len[base + q]] - S.start[c0] + 63) / 64;
      }
      local += nc[q];
    }
    int32_t total;
    int32_t ex = block_scan_256(local, total, wsum) + carry;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      if (base + q < P.nrows) {
        S.row_chunk_off[base + q] = ex;
        for (int c = 0; c < nc[q]; ++c) S.chunk_row[ex + c] = base + q;
      }
      ex += nc[q];
    }
    carry += total;
  }
  if (threadIdx.x == 0) S.row_chunk_off[P.nrows] = carry;
}

__device__ __forceinline__ void sort_scatter(const DevParams& P, const DeviceState& S, int item) {
  for (int q = 0; q < kSortItem / kSortThreads; ++q) {
    const int i = item * kSortItem + q * kSortThreads + (int)threadIdx.x;
    if (i < P.n) S.unsorted[S.start[S.key[i]] + S.slot[i]] = i;
  }
}

// Rank inside the cell by index (stable order) and move the state there.
__device__ __forceinline__ void sort_place(const DevParams& P, const DeviceState& S, int item,
                                           int items) {
  const int64_t n = P.n;
  const int dim = P.dim;
  const int64_t c0 = (int64_t)P.ncell * item / items, c1 = (int64_t)P.ncell * (item + 1) / items;
  for (int64_t c = c0 + threadIdx.x; c < c1; c += kSortThreads) S.count[c] = 0;
  for (int qq = 0; qq < kSortItem / kSortThreads; ++qq) {
    const int i = item * kSortItem + qq * kSortThreads + (int)threadIdx.x;
    if (i >= P.n) continue;
    const int32_t k = S.key[i];
    const int32_t s = S.start[k], e = S.start[k + 1];
    int32_t r = 0;
    for (int32_t q = s; q < e; ++q) r += S.unsorted[q] < i ? 1 : 0;
    const int32_t p = s + r;
    double xv[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < dim; ++d) {
      xv[d] = S.x[d * n + i];
      S.x_alt[d * n + p] = xv[d];
      S.v_alt[d * n + p] = S.v[d * n + i];
    }
    S.m_alt[p] = S.m[i];
    S.pid_alt[p] = S.pid[i];
    S.perm_alt[p] = S.perm[i];
    if (P.ncoll) {
      // colloids: species id moves with the particle; the slot of each upload
      // index locates the boundary particles of a colloid
      S.sid_alt[p] = S.sid[i];
      S.slot_of[S.perm[i]] = p;
    }
    const int rq = S.rep[i];
    S.rep_alt[p] = rq;
    S.key_sorted[p] = k;
    if (!P.newtonian) {
      const int d2 = dim * dim;
      for (int q = 0; q < d2; ++q) S.ct_alt[q * n + p] = S.ct[q * n + i];
    }
    // FP32 position relative to the lower corner of the own cell, the cell's
    // x index in w (records of the neighbour scan)
    const RepGeom& g = S.geo[rq];
    const int kl = k - g.cell_base;
    const int cx = kl % g.nm[0];
    const int cy = (kl / g.nm[0]) % g.nm[1];
    const int cz = kl / (g.nm[0] * g.nm[1]);
    S.xa[p] = make_float4((float)(xv[0] - (g.lo[0] + (double)cx * g.cs[0])),
                          (float)(xv[1] - (g.lo[1] + (double)cy * g.cs[1])),
                          dim == 3 ? (float)(xv[2] - (g.lo[2] + (double)cz * g.cs[2])) : 0.f,
                          __int_as_float(cx));
  }
}

// The sorted state back from the *_alt buffers into the primary ones, the
// sorted positions into x_ref (the positions of the lists' build) and into
// what the walks gather.
__device__ __forceinline__ void sort_back(const DevParams& P, const DeviceState& S, int item) {
  const int64_t n = P.n;
  for (int qq = 0; qq < kSortItem / kSortThreads; ++qq) {
    const int i = item * kSortItem + qq * kSortThreads + (int)threadIdx.x;
    if (i >= P.n) continue;
    double xv[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < P.dim; ++d) {
      xv[d] = S.x_alt[d * n + i];
      S.x[d * n + i] = xv[d];
      S.x_ref[d * n + i] = xv[d];
      S.v[d * n + i] = S.v_alt[d * n + i];
    }
    const int32_t pid = S.pid_alt[i], rq = S.rep_alt[i];
    if (P.mixed) {
      const RepGeom& g = S.geo[rq];
      S.xq[i] = make_uint4(fixed_position(g, 0, xv[0]), fixed_position(g, 1, xv[1]),
                           P.dim == 3 ? fixed_position(g, 2, xv[2]) : 0u, (uint32_t)pid);
    } else {
      reinterpret_cast<double2*>(S.rec64)[i] = make_double2(xv[0], xv[1]);
    }
    S.m[i] = S.m_alt[i];
    S.pid[i] = pid;
    S.perm[i] = S.perm_alt[i];
    S.rep[i] = rq;
    if (!P.newtonian) {
      const int d2 = P.dim * P.dim;
      for (int q = 0; q < d2; ++q) S.ct[q * n + i] = S.ct_alt[q * n + i];
    }
    if (P.ncoll) S.sid[i] = S.sid_alt[i];
  }
}

__device__ __forceinline__ void sort_item(const DevParams& P, const DeviceState& S,
                                          const SortPlan& plan, int phase, int item,
                                          int32_t* wsum) {
  switch (phase) {
    case kKeys: sort_keys(P, S, item); break;
    case kSums: sort_sums(P, S, item, wsum); break;
    case kStarts: sort_starts(P, S, item, wsum); break;
    case kScatter:
      if (item == 0)
        sort_rows(P, S, wsum);
      else
        sort_scatter(P, S, item - 1);
      break;
    case kPlace: sort_place(P, S, item, plan.items[kPlace]); break;
    default: sort_back(P, S, item); break;
  }
}

// One launch per phase: for callers that may overlap on the same buffers
// (k_sort_chain's counters would not survive that).
__global__ __launch_bounds__(kSortThreads) void k_sort_phase(DevParams P, DeviceState S,
                                                             SortPlan plan, int phase) {
  __shared__ int32_t wsum[4];
  sort_item(P, S, plan, phase, blockIdx.x, wsum);
}

// Whether the lists are rebuilt this step: a particle moved more than skin / 2
// since their build (a pair then may have closed in by more than the skin), or
// a build is pending (a sort whose lists no density pass has built yet).
__device__ __forceinline__ bool lists_outdated(const DevParams& P, const DeviceState& S,
                                               bool& moved) {
  const double d2 = __longlong_as_double((long long)S.disp[0]);
  double lim = P.half_skin2;
  moved = false;
  if (P.le_g >= 0) {
    // sheared faces: the copies across a face move by |v_upper - v_lower|
    // per unit time against the box, so a pair across it may have closed
    // in by that drift since the build on top of the particles' own
    // displacements: the lists hold while 2 max |dx| + drift < skin.  A
    // list that overflowed rebuilds every step (the rescans then always
    // see the positions of a build).
    const double drift = fabs(P.le_vhi - P.le_vlo) * fabs(S.time_dev[1] - S.time_dev[3]);
    const double room = 0.5 * (P.skin - drift);
    lim = room > 0.0 ? room * room : -1.0;
    moved = S.gate[2] != 0;
  }
  moved = moved || d2 > lim;
  return moved || S.gate[0] != 0;
}

// The whole sort in one launch.  Launched one by one its 13 kernels cost a
// step 2.6 to 4.5 us each, most of a small box's step, and with Verlet lists
// nearly all of those launches return at once (with the gate, the list flags
// and the step advance folded in as well: 12^3 box 76 -> 47 us per step,
// 37 x 29 x 41 126 -> 87, 64 x 64 81 -> 58).  Workgroups draw items in phase order
// from a ticket counter; an item first waits until every item of the phase
// before it is done.  Whoever waits holds a later ticket than what it waits
// for, and tickets are only drawn by running workgroups, so the oldest
// unfinished item never waits on one that has not started: the waits end
// whatever the number of workgroups on the GPU.
//
// ctl: [0] tickets, [1 + phase] items done, [7] workgroups that left; zero
// between launches (the last workgroup to leave clears them).
// mode 0: per-step lists.  1 (Verlet lists): sorts when the lists are
// outdated.  2 (Verlet lists): sorts in any case.  advance: also one marching
// step (nothing else here reads the step).
__global__ __launch_bounds__(kSortThreads) void k_sort_chain(DevParams P, DeviceState S,
                                                             SortPlan plan, int mode,
                                                             int advance) {
  __shared__ int32_t wsum[4];
  __shared__ int32_t drawn;
  bool moved = mode == 2;
  if (advance && blockIdx.x == 0 && threadIdx.x == 0) advance_step(S.step_dev, S.time_dev, P.dt);
  if (mode == 1 && !lists_outdated(P, S, moved)) return;
  int32_t* ctl = S.sort_ctl;
  int total = 0;
  for (int p = 0; p < kSortPhases; ++p) total += plan.items[p];
  int ready = -1;  // phases up to this one are known to be done
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) drawn = atomicAdd(&ctl[0], 1);
    __syncthreads();
    int item = drawn;
    if (item >= total) break;
    int phase = 0;
    while (item >= plan.items[phase]) item -= plan.items[phase++];
    if (phase - 1 > ready) {
      // (a phase without items is done; the phases before the last one with
      // items were done when that one began)
      int before = phase - 1;
      while (before >= 0 && plan.items[before] == 0) --before;
      if (before >= 0) {
        if (threadIdx.x == 0) {
          while (__hip_atomic_load(&ctl[1 + before], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
                 plan.items[before])
            __builtin_amdgcn_s_sleep(2);
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        __syncthreads();
      }
      ready = phase - 1;
    }
    sort_item(P, S, plan, phase, item, wsum);
    // every wave's stores have reached the L2 before thread 0 writes it back
    // (a workgroup barrier alone does not wait for them)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __hip_atomic_fetch_add(&ctl[1 + phase], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (threadIdx.x != 0) return;
  if (atomicAdd(&ctl[7], 1) != (int)gridDim.x - 1) return;
  // the last workgroup: every other one has read what is written here
  for (int q = 0; q < 8; ++q) ctl[q] = 0;
  if (mode == 0) return;
  // gate[0]: the next density pass builds the lists; gate[1] counts the
  // builds; gate[2], set by the build, flags lists that overflowed
  S.gate[0] = 1;
  if (moved) {
    S.gate[1] += 1;
    S.gate[2] = 0;
    S.disp[0] = 0ull;
  }
}

// ---------------------------------------------------------------------
// PPM's cell list on PPM's grid (cell edge >= 1.0001 cut_off), in upload
// indices: the order inside a cell is ascending upload index, which is
// what ppm_util_rank3d produces for particles stored in upload order.
// ---------------------------------------------------------------------
__global__ void k_ref_key(DevParams P, const double* __restrict__ x, int32_t* __restrict__ key,
                          int32_t* __restrict__ slot, int32_t* __restrict__ count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  const int64_t n = P.n;
  int cx = cell_coord(x[i], P.min_phys[0], P.rd_ref[0], P.min_phys[0] + P.length[0], P.nm_ref[0]);
  int cy = cell_coord(x[n + i], P.min_phys[1], P.rd_ref[1], P.min_phys[1] + P.length[1],
                      P.nm_ref[1]);
  int cz = P.dim == 3 ? cell_coord(x[2 * n + i], P.min_phys[2], P.rd_ref[2],
                                   P.min_phys[2] + P.length[2], P.nm_ref[2])
                      : 0;
  int32_t k = cx + P.nm_ref[0] * (cy + P.nm_ref[1] * cz);
  key[i] = k;
  slot[i] = atomicAdd(&count[k], 1);
}

__global__ void k_ref_rank(int n, const int32_t* __restrict__ key,
                           const int32_t* __restrict__ start,
                           const int32_t* __restrict__ unsorted,
                           const int32_t* __restrict__ perm, int32_t* __restrict__ lpdx) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int32_t k = key[i];
  int32_t s = start[k], e = start[k + 1];
  int32_t me = perm[i], r = 0;
  for (int32_t q = s; q < e; ++q) r += perm[unsorted[q]] < me ? 1 : 0;
  lpdx[s + r] = me;
}

// ---------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------
static inline int blocks_for(int64_t n, int bs) { return (int)((n + bs - 1) / bs); }

void launch_fill_i32(hipStream_t s, int32_t* a, int32_t v, int64_t n) {
  if (n <= 0) return;
  int nb = blocks_for(n, 256);
  if (nb > 4096) nb = 4096;
  hipLaunchKernelGGL(k_fill_i32, dim3(nb), dim3(256), 0, s, a, v, n);
}

void launch_fill_f64(hipStream_t s, double* a, double v, int64_t n) {
  if (n <= 0) return;
  int nb = blocks_for(n, 256);
  if (nb > 4096) nb = 4096;
  hipLaunchKernelGGL(k_fill_f64, dim3(nb), dim3(256), 0, s, a, v, n);
}

// Workgroups of the chain: up to four per CU, no more than its longest phase
// has items.
static inline dim3 sort_grid(const SortPlan& plan) {
  int most = 1;
  for (int p = 0; p < kSortPhases; ++p) most = std::max(most, plan.items[p]);
  return dim3(std::min(most, 1024));
}

void launch_sort(hipStream_t s, const DevParams& P, const DeviceState& S, SortKind kind,
                 bool advance) {
  const bool keys = kind != SortKind::kStepKeysDone;
  const bool verlet = kind == SortKind::kVerletGated || kind == SortKind::kVerletForced;
  const SortPlan plan = sort_plan(P, keys, verlet);
  const int mode = !verlet ? 0 : (kind == SortKind::kVerletGated ? 1 : 2);
  hipLaunchKernelGGL(k_sort_chain, sort_grid(plan), dim3(kSortThreads), 0, s, P, S, plan, mode,
                     advance ? 1 : 0);
}

void launch_sort_phases(hipStream_t s, const DevParams& P, const DeviceState& S, bool copy_back) {
  const SortPlan plan = sort_plan(P, true, copy_back);
  for (int p = 0; p < kSortPhases; ++p)
    if (plan.items[p] > 0)
      hipLaunchKernelGGL(k_sort_phase, dim3(plan.items[p]), dim3(kSortThreads), 0, s, P, S, plan,
                         p);
}

void launch_reference_cells(hipStream_t s, const DevParams& P, const DeviceState& S) {
  const int n = P.n;
  launch_fill_i32(s, S.rcount, 0, P.ncell_ref);
  hipLaunchKernelGGL(k_ref_key, dim3(blocks_for(n, 256)), dim3(256), 0, s, P, S.x, S.rkey,
                     S.rslot, S.rcount);
  launch_exclusive_scan(s, S.rcount, S.rstart, P.ncell_ref, S.scan_tmp);
  hipLaunchKernelGGL(k_scatter, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, S.rkey, S.rslot,
                     S.rstart, S.runsorted);
  hipLaunchKernelGGL(k_ref_rank, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, S.rkey, S.rstart,
                     S.runsorted, S.perm, S.rlpdx);
}

}  // namespace sdpd
