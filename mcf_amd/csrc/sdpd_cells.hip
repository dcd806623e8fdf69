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
//   keys     cell key, slot and histogram       ITEM particles per item
//   sums     sums of 4096 cell counts           one tile per item
//   starts   first particle of every cell       one tile per item, which adds
//                                               up the sums of the tiles before
//   scatter  unsorted[start[key] + slot] = i    ITEM particles; item 0 is the
//                                               pair kernels' work map
//   place    rank in the cell, state moved to the *_alt buffers, cell counts
//            cleared for the next sort          ITEM particles
//   back     the state copied back, with x_ref and the walks' positions
//                                               ITEM particles (Verlet lists)
// The counts are zero between sorts.
constexpr int kSortThreads = 256;    // of a launch per phase, and particles per item
constexpr int kChainThreads = 1024;  // of the one launch, likewise
enum SortPhase { kKeys = 0, kSums, kStarts, kScatter, kPlace, kBack, kSortPhases };

struct SortPlan {
  int32_t items[kSortPhases];
};

static SortPlan sort_plan(const DevParams& P, int item, bool keys, bool copy_back) {
  const int32_t blocks = (P.n + item - 1) / item;
  const int32_t tiles = (P.ncell + kScanTile - 1) / kScanTile;
  return {{keys ? blocks : 0, tiles, tiles, blocks + 1, blocks, copy_back ? blocks : 0}};
}

// exclusive scan over the workgroup's T threads
template <int T>
__device__ __forceinline__ int32_t block_scan(int32_t v, int32_t& total, int32_t* wsum) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t t = __shfl_up(incl, off, 64);
    if (lane >= off) incl += t;
  }
  if (lane == 63) wsum[wid] = incl;
  __syncthreads();
  int32_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < T / 64; ++w) {
    before += w < wid ? wsum[w] : 0;
    total += wsum[w];
  }
  __syncthreads();
  return before + incl - v;
}

template <int T, int ITEM>
__device__ __forceinline__ void sort_keys(const DevParams& P, const DeviceState& S, int item) {
  const int64_t n = P.n;
#pragma unroll
  for (int q = 0; q < ITEM / T; ++q) {
    const int i0 = item * ITEM + q * T + (int)threadIdx.x;
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

template <int T>
__device__ __forceinline__ void sort_sums(const DevParams& P, const DeviceState& S, int item,
                                          int32_t* wsum) {
  const int64_t base = (int64_t)item * kScanTile + threadIdx.x * (kScanTile / T);
  int32_t local = 0;
#pragma unroll
  for (int q = 0; q < kScanTile / T; ++q)
    if (base + q < P.ncell) local += S.count[base + q];
  int32_t total;
  (void)block_scan<T>(local, total, wsum);
  if (threadIdx.x == 0) S.scan_tmp[item] = total;
}

template <int T>
__device__ __forceinline__ void sort_starts(const DevParams& P, const DeviceState& S, int item,
                                            int32_t* wsum) {
  int32_t part = 0, before;
  for (int t = threadIdx.x; t < item; t += T) part += S.scan_tmp[t];
  (void)block_scan<T>(part, before, wsum);
  constexpr int kPer = kScanTile / T;
  const int64_t base = (int64_t)item * kScanTile + threadIdx.x * kPer;
  int32_t v[kPer], local = 0;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    v[q] = base + q < P.ncell ? S.count[base + q] : 0;
    local += v[q];
  }
  int32_t total;
  int32_t ex = block_scan<T>(local, total, wsum) + before;
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
template <int T>
__device__ __forceinline__ void sort_rows(const DevParams& P, const DeviceState& S,
                                          const int32_t* start, int32_t* wsum) {
  constexpr int kPer = 4;
  int32_t carry = 0;
  for (int r0 = 0; r0 < P.nrows; r0 += kPer * T) {
    const int base = r0 + (int)threadIdx.x * kPer;
    int32_t nc[kPer], local = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      nc[q] = 0;
      if (base + q < P.nrows) {
        const int c0 = S.row_cell[base + q];
        nc[q] = (start[c0 + S.row_len[base + q]] - start[c0] + 63) / 64;
      }
      local += nc[q];
    }
    int32_t total;
    int32_t ex = block_scan<T>(local, total, wsum) + carry;
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

template <int T, int ITEM>
__device__ __forceinline__ void sort_scatter(const DevParams& P, const DeviceState& S, int item) {
#pragma unroll
  for (int q = 0; q < ITEM / T; ++q) {
    const int i = item * ITEM + q * T + (int)threadIdx.x;
    if (i < P.n) S.unsorted[S.start[S.key[i]] + S.slot[i]] = i;
  }
}

// A particle's state in registers: every load is issued before the first
// store (the buffers may alias as far as the compiler knows).
struct Moved {
  double x[3], v[3], m, ct[9];
  int32_t pid, perm, rep, sid;
};
__device__ __forceinline__ Moved load_moved(const DevParams& P, int i, const double* x,
                                            const double* v, const double* m, const double* ct,
                                            const int32_t* pid, const int32_t* perm,
                                            const int32_t* rep, const int32_t* sid) {
  const int64_t n = P.n;
  Moved a;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    a.x[d] = d < P.dim ? x[d * n + i] : 0.0;
    a.v[d] = d < P.dim ? v[d * n + i] : 0.0;
  }
  a.m = m[i];
  a.pid = pid[i];
  a.perm = perm[i];
  a.rep = rep[i];
  a.sid = P.ncoll ? sid[i] : 0;
  if (!P.newtonian) {
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (q < P.dim * P.dim) a.ct[q] = ct[q * n + i];
  }
  return a;
}
__device__ __forceinline__ void store_moved(const DevParams& P, int p, const Moved& a, double* x,
                                            double* v, double* m, double* ct, int32_t* pid,
                                            int32_t* perm, int32_t* rep, int32_t* sid) {
  const int64_t n = P.n;
#pragma unroll
  for (int d = 0; d < 3; ++d)
    if (d < P.dim) {
      x[d * n + p] = a.x[d];
      v[d * n + p] = a.v[d];
    }
  m[p] = a.m;
  pid[p] = a.pid;
  perm[p] = a.perm;
  rep[p] = a.rep;
  if (P.ncoll) sid[p] = a.sid;
  if (!P.newtonian) {
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (q < P.dim * P.dim) ct[q * n + p] = a.ct[q];
  }
}

// FP32 position relative to the lower corner of the own cell, the cell's x
// index in w (records of the neighbour scan).
__device__ __forceinline__ float4 cell_record(const DevParams& P, const RepGeom& g, int32_t k,
                                              const double* x) {
  const int kl = k - g.cell_base;
  const int cx = kl % g.nm[0];
  const int cy = (kl / g.nm[0]) % g.nm[1];
  const int cz = kl / (g.nm[0] * g.nm[1]);
  return make_float4((float)(x[0] - (g.lo[0] + (double)cx * g.cs[0])),
                     (float)(x[1] - (g.lo[1] + (double)cy * g.cs[1])),
                     P.dim == 3 ? (float)(x[2] - (g.lo[2] + (double)cz * g.cs[2])) : 0.f,
                     __int_as_float(cx));
}

// What the walks gather of the position of slot p, and x_ref.
__device__ __forceinline__ void store_positions(const DevParams& P, const DeviceState& S,
                                                const RepGeom& g, int p, const Moved& a) {
  const int64_t n = P.n;
  if (P.mixed) {
    S.xq[p] = make_uint4(fixed_position(g, 0, a.x[0]), fixed_position(g, 1, a.x[1]),
                         P.dim == 3 ? fixed_position(g, 2, a.x[2]) : 0u, (uint32_t)a.pid);
  } else {
    reinterpret_cast<double2*>(S.rec64)[p] = make_double2(a.x[0], a.x[1]);
  }
  if (S.x_ref) {
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (d < P.dim) S.x_ref[d * n + p] = a.x[d];
  }
}

// Rank inside the cell by index (stable order) and move the state there.
template <int T, int ITEM>
__device__ __forceinline__ void sort_place(const DevParams& P, const DeviceState& S, int item,
                                           int items) {
  const int64_t c0 = (int64_t)P.ncell * item / items, c1 = (int64_t)P.ncell * (item + 1) / items;
  for (int64_t c = c0 + threadIdx.x; c < c1; c += T) S.count[c] = 0;
  for (int qq = 0; qq < ITEM / T; ++qq) {
    const int i = item * ITEM + qq * T + (int)threadIdx.x;
    if (i >= P.n) continue;
    const int32_t k = S.key[i];
    const Moved a = load_moved(P, i, S.x, S.v, S.m, S.ct, S.pid, S.perm, S.rep, S.sid);
    const int32_t s = S.start[k], e = S.start[k + 1];
    int32_t r = 0;
    for (int32_t q = s; q < e; q += 8) {
      int32_t u[8];
#pragma unroll
      for (int w = 0; w < 8; ++w) u[w] = S.unsorted[min(q + w, e - 1)];
#pragma unroll
      for (int w = 0; w < 8; ++w) r += (q + w < e && u[w] < i) ? 1 : 0;
    }
    const int32_t p = s + r;
    const float4 xa = cell_record(P, S.geo[a.rep], k, a.x);
    store_moved(P, p, a, S.x_alt, S.v_alt, S.m_alt, S.ct_alt, S.pid_alt, S.perm_alt, S.rep_alt,
                S.sid_alt);
    S.key_sorted[p] = k;
    S.xa[p] = xa;
    // (the slot of each upload index locates the boundary particles of a
    // colloid)
    if (P.ncoll) S.slot_of[a.perm] = p;
  }
}

// The sorted state back from the *_alt buffers into the primary ones, the
// sorted positions into x_ref (the positions of the lists' build; not kept by
// a single evaluation) and into what the walks gather.
template <int T, int ITEM>
__device__ __forceinline__ void sort_back(const DevParams& P, const DeviceState& S, int item) {
  for (int qq = 0; qq < ITEM / T; ++qq) {
    const int i = item * ITEM + qq * T + (int)threadIdx.x;
    if (i >= P.n) continue;
    const Moved a = load_moved(P, i, S.x_alt, S.v_alt, S.m_alt, S.ct_alt, S.pid_alt, S.perm_alt,
                               S.rep_alt, S.sid_alt);
    store_positions(P, S, S.geo[a.rep], i, a);
    store_moved(P, i, a, S.x, S.v, S.m, S.ct, S.pid, S.perm, S.rep, S.sid);
  }
}

template <int T, int ITEM>
__device__ __forceinline__ void sort_item(const DevParams& P, const DeviceState& S,
                                          const SortPlan& plan, int phase, int item,
                                          int32_t* wsum) {
  switch (phase) {
    case kKeys: sort_keys<T, ITEM>(P, S, item); break;
    case kSums: sort_sums<T>(P, S, item, wsum); break;
    case kStarts: sort_starts<T>(P, S, item, wsum); break;
    case kScatter:
      if (item == 0)
        sort_rows<T>(P, S, S.start, wsum);
      else
        sort_scatter<T, ITEM>(P, S, item - 1);
      break;
    case kPlace: sort_place<T, ITEM>(P, S, item, plan.items[kPlace]); break;
    default: sort_back<T, ITEM>(P, S, item); break;
  }
}

// One launch per phase: for callers that may overlap on the same buffers
// (k_sort_chain's counters would not survive that), and for lists rebuilt every
// step.  ADVANCE: also one marching step.
template <bool ADVANCE>
__global__ __launch_bounds__(kSortThreads) void k_sort_phase(DevParams P, DeviceState S,
                                                             SortPlan plan, int phase) {
  __shared__ int32_t wsum[kSortThreads / 64];
  if (ADVANCE && blockIdx.x == 0 && threadIdx.x == 0) advance_step(S.step_dev, S.time_dev, P.dt);
  sort_item<kSortThreads, kSortThreads>(P, S, plan, phase, blockIdx.x, wsum);
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

// After a sort for Verlet lists.  gate[0]: the next density pass builds the
// lists; gate[1] counts the builds; gate[2], set by the build, flags lists that
// overflowed.
__device__ __forceinline__ void set_gate(const DeviceState& S, bool moved) {
  S.gate[0] = 1;
  if (moved) {
    S.gate[1] += 1;
    S.gate[2] = 0;
    S.disp[0] = 0ull;
  }
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
// A workgroup counts its items of a phase in one go, before it waits for the
// next phase or ends: the count needs its XCD's L2 written back, and with a
// write-back per item, and workgroups of 256, a rebuild's sort took 893 us at
// 128^3, 490 at 100^3, 140 at 45^3 and 48 at 30^3 (349, 188, 50 and 37 now).  For
// the same reason the workgroups are large and few: 128 of 1024 threads, 256
// beyond 2^20 particles (64^3 80 us with 128, 91 with 256; 128^3 384 and 349).
//
// ctl: [0] tickets, [1 + phase] items done, [7] workgroups that left; zero
// between launches (the last workgroup to leave clears them).
// Verlet lists only.  mode 1: sorts when the lists are outdated, 2: in any case.
// advance: also one marching step (nothing else here reads the step).
__global__ __launch_bounds__(kChainThreads) void k_sort_chain(DevParams P, DeviceState S,
                                                             SortPlan plan, int mode,
                                                             int advance) {
  constexpr int T = kChainThreads;
  __shared__ int32_t wsum[T / 64];
  __shared__ int32_t drawn;
  bool moved = mode == 2;
  if (advance && blockIdx.x == 0 && threadIdx.x == 0) advance_step(S.step_dev, S.time_dev, P.dt);
  if (mode == 1 && !lists_outdated(P, S, moved)) return;
  int32_t* ctl = S.sort_ctl;
  int ready = -1;  // phases up to this one are known to be done
  int held = 0, of = 0;  // items of phase `of` done here and not yet counted
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) drawn = atomicAdd(&ctl[0], 1);
    __syncthreads();
    int item = drawn, phase = 0;
    while (phase < kSortPhases && item >= plan.items[phase]) item -= plan.items[phase++];
    if (held > 0 && phase != of) {
      // every wave's stores have reached the L2 before thread 0 writes it back
      // (a workgroup barrier alone does not wait for them)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __hip_atomic_fetch_add(&ctl[1 + of], held, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      held = 0;
    }
    if (phase == kSortPhases) break;
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
    sort_item<T, T>(P, S, plan, phase, item, wsum);
    held += 1;
    of = phase;
  }
  if (threadIdx.x != 0) return;
  // (this workgroup's counts are in before it is counted out)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (atomicAdd(&ctl[7], 1) != (int)gridDim.x - 1) return;
  // the last workgroup: every other one has read what is written here
  for (int q = 0; q < 8; ++q) ctl[q] = 0;
  set_gate(S, moved);
}

// The sort of a small box: every workgroup counts all the cells for itself in
// LDS, so that the phases up to the placing need no exchange, and places 256
// particles; the last one to finish copies the state back.  Nothing waits, and
// ctl[0] alone is shared.  64 x 64 particles: 20 us, 51 with k_sort_chain,
// 39 with the whole sort in one workgroup (one CU's issue rate).
// mode: k_sort_chain's, without the gate 3 as 2, and 0 and 4 for lists rebuilt
// every step; keys_done: the step boundary has counted the cells in S.count, which
// are cleared.
constexpr int kSmallThreads = 1024;
constexpr int kSmallPer = 4;
constexpr int kSmallParticles = kSmallThreads * kSmallPer;
constexpr int kSmallCellsPer = 8;
constexpr int kSmallCells = kSmallThreads * kSmallCellsPer;
constexpr int kSmallOwn = 256;
__global__ __launch_bounds__(kSmallThreads) void k_sort_small(DevParams P, DeviceState S, int mode,
                                                              int keys_done, int advance) {
  __shared__ int32_t wsum[kSmallThreads / 64];
  __shared__ int32_t start[kSmallCells + 1];
  __shared__ int32_t unsorted[kSmallParticles];
  __shared__ int32_t arrived;
  const int tid = threadIdx.x;
  const int64_t n = P.n;
  bool moved = mode == 2;
  if (advance && blockIdx.x == 0 && tid == 0) advance_step(S.step_dev, S.time_dev, P.dt);
  if (mode == 1 && !lists_outdated(P, S, moved)) return;
  double x[kSmallPer][3];
  int32_t rep[kSmallPer], key[kSmallPer], slot[kSmallPer];
#pragma unroll
  for (int q = 0; q < kSmallPer; ++q) {
    const int i = min(q * kSmallThreads + tid, P.n - 1);
    rep[q] = S.rep[i];
#pragma unroll
    for (int d = 0; d < 3; ++d) x[q][d] = d < P.dim ? S.x[d * n + i] : 0.0;
  }
  // the particles that this workgroup places, 256 of its threads one each
  constexpr int kOwners = kSmallThreads / kSmallOwn;
  const int mine = (int)blockIdx.x / kOwners;  // which of a thread's particles
  const int own = mine * kSmallThreads + tid;
  const bool owner = tid / kSmallOwn == (int)blockIdx.x % kOwners && own < P.n;
  Moved a;
  if (owner) a = load_moved(P, own, S.x, S.v, S.m, S.ct, S.pid, S.perm, S.rep, S.sid);
  for (int c = tid; c <= P.ncell; c += kSmallThreads) start[c] = 0;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSmallPer; ++q) {
    key[q] = cell_key_geo(S.geo[rep[q]], P.dim, x[q][0], x[q][1], x[q][2]);
    slot[q] = q * kSmallThreads + tid < P.n ? atomicAdd(&start[key[q]], 1) : 0;
  }
  __syncthreads();
  {
    int32_t v[kSmallCellsPer], local = 0, total;
    const int c0 = tid * kSmallCellsPer;
#pragma unroll
    for (int u = 0; u < kSmallCellsPer; ++u) {
      v[u] = c0 + u < P.ncell ? start[c0 + u] : 0;
      local += v[u];
    }
    int32_t ex = block_scan<kSmallThreads>(local, total, wsum);
#pragma unroll
    for (int u = 0; u < kSmallCellsPer; ++u) {
      if (c0 + u < P.ncell) {
        start[c0 + u] = ex;
        if (blockIdx.x == 0) S.start[c0 + u] = ex;
      }
      ex += v[u];
    }
    if (tid == 0) start[P.ncell] = total;
    if (tid == 0 && blockIdx.x == 0) S.start[P.ncell] = total;
  }
  __syncthreads();
  int32_t k = 0;
#pragma unroll
  for (int q = 0; q < kSmallPer; ++q) {
    const int i = q * kSmallThreads + tid;
    if (i < P.n) unsorted[start[key[q]] + slot[q]] = i;
    if (q == mine) k = key[q];
  }
  if (blockIdx.x == 0) sort_rows<kSmallThreads>(P, S, start, wsum);
  __syncthreads();
  if (owner) {
    const int s = start[k], e = start[k + 1];
    int p = s;
    for (int w = s; w < e; ++w) p += unsorted[w] < own ? 1 : 0;
    const float4 xa = cell_record(P, S.geo[a.rep], k, a.x);
    store_moved(P, p, a, S.x_alt, S.v_alt, S.m_alt, S.ct_alt, S.pid_alt, S.perm_alt, S.rep_alt,
                S.sid_alt);
    S.key_sorted[p] = k;
    S.xa[p] = xa;
    if (P.ncoll) S.slot_of[a.perm] = p;
  }
  // (as in k_sort_chain)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    arrived = __hip_atomic_fetch_add(&S.sort_ctl[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  if (arrived != (int)gridDim.x - 1) return;
  if (mode != 0 && mode != 4)
    for (int q = 0; q < kSmallPer; ++q) sort_back<kSmallThreads, kSmallThreads>(P, S, q);
  if (keys_done)
    for (int c = tid; c < P.ncell; c += kSmallThreads) S.count[c] = 0;
  if (tid != 0) return;
  S.sort_ctl[0] = 0;
  if (mode == 1 || mode == 2) set_gate(S, moved);
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

static inline bool sort_small(const DevParams& P) {
  return P.n <= kSmallParticles && P.ncell <= kSmallCells;
}
static inline dim3 small_grid(const DevParams& P) {
  return dim3((P.n + kSmallOwn - 1) / kSmallOwn);
}

// Workgroups of the chain, no more than its longest phase has items.
static inline dim3 sort_grid(const DevParams& P, const SortPlan& plan) {
  int most = 1;
  for (int p = 0; p < kSortPhases; ++p) most = std::max(most, plan.items[p]);
  return dim3(std::min(most, P.n > (1 << 20) ? 256 : 128));
}

// (Lists rebuilt every step always sort: nothing to gain from a launch that may
// return at once.  us with the chain and with a launch per phase: 30^3 25 and 24,
// 45^3 31 and 26, 64^3 47 and 35, 100^3 103 and 81, 128^3 180 and 139.)
static void launch_phases(hipStream_t s, const DevParams& P, const DeviceState& S, bool keys,
                          bool copy_back, bool advance) {
  const SortPlan plan = sort_plan(P, kSortThreads, keys, copy_back);
  for (int p = 0; p < kSortPhases; ++p)
    if (plan.items[p] > 0) {
      const auto kernel = advance ? k_sort_phase<true> : k_sort_phase<false>;
      hipLaunchKernelGGL(kernel, dim3(plan.items[p]), dim3(kSortThreads), 0, s, P, S, plan, p);
      advance = false;
    }
}

void launch_sort(hipStream_t s, const DevParams& P, const DeviceState& S, SortKind kind,
                 bool advance) {
  const bool keys = kind != SortKind::kStepKeysDone;
  const bool verlet = kind == SortKind::kVerletGated || kind == SortKind::kVerletForced;
  const int mode = !verlet ? 0 : (kind == SortKind::kVerletGated ? 1 : 2);
  if (sort_small(P)) {
    hipLaunchKernelGGL(k_sort_small, small_grid(P), dim3(kSmallThreads), 0, s, P, S, mode,
                       keys ? 0 : 1, advance ? 1 : 0);
  } else if (!verlet) {
    launch_phases(s, P, S, keys, false, advance);
  } else {
    const SortPlan plan = sort_plan(P, kChainThreads, true, true);
    hipLaunchKernelGGL(k_sort_chain, sort_grid(P, plan), dim3(kChainThreads), 0, s, P, S, plan, mode,
                       advance ? 1 : 0);
  }
}

void launch_sort_phases(hipStream_t s, const DevParams& P, const DeviceState& S, bool copy_back) {
  if (sort_small(P)) {
    hipLaunchKernelGGL(k_sort_small, small_grid(P), dim3(kSmallThreads), 0, s, P, S,
                       copy_back ? 3 : 4, 0, 0);
    return;
  }
  launch_phases(s, P, S, true, copy_back, false);
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
