// sdpd_pair.hip -- K2 density + equation of state and K4 pair forces
// (gfx950), FP64 and mixed precision.
//
// Replaces the two hot loops of the reference: particles_compute_density
// (particles_compute_density.F90:578-867) and particles_compute_interaction
// (particles_compute_interaction.F90:618-911 with pp_interaction.inc,
// pp_interaction_ff.inc, pp_vgt_ip.inc and rhs_force_ff_*).  The reference
// visits each unordered pair once in a half stencil and adds the result to
// both particles and to periodic ghost copies that are folded back later.
// Here every particle gathers over the cells around its own, with the
// periodic image applied per stencil segment, and writes only its own
// sums: no atomics, no ghosts, identical results run to run.
//
// Work decomposition.  The sort grid has half of PPM's cell edge, so the
// neighbours of a particle lie in the 5 x 5 x 5 (2D: 5 x 5) block of cells
// around its own.  One wavefront takes a chunk of at most 64 consecutive
// particles of one (y, z) row of cells, so all its lanes share the 25
// (2D: 5) stencil rows.  For each stencil row the wave stages the union of
// its lanes' candidate cells into LDS with coalesced loads -- laid out in
// "virtual cell" order, where the cells seen across a periodic x face
// follow the row with their image shift -- and every lane scans the five
// cells around its own from LDS.
//
// Cut-off decision (both modes): r^2 in FP32 on positions relative to the
// cell corner; a candidate within a band around rc^2 wider than the FP32
// error bound is re-decided in FP64 exactly as the reference forms it
// (pp_interaction.inc:37-46) with the reference's periodic image
// convention.  Neighbour sets are therefore bit-exact in both modes.
//
// The density pass appends the accepted neighbours of every particle to a
// per-lane LDS list, evaluates the density terms whenever the lists fill
// up, and stores the lists of a chunk as one block of groups of 8 entries
// per lane: every store fills whole 32-byte sectors and the force pass of
// the same step (positions unchanged) reads 2 KB contiguous per group.
#include <type_traits>

#include "sdpd_kernels.h"
#include "sdpd_window.h"

namespace sdpd {

constexpr int kWave = 64;
// Defaults of the two tunable shapes of the candidate scan (the density kernel of
// lists rebuilt every step is instantiated for the autotuner's other choices too):
constexpr int kBuf = 16;          // LDS list entries per lane between flushes (>= 10)
constexpr int kTile = 224;        // staged candidate records per stencil row batch
constexpr int kCodeShift = 25;    // list entry = j | (stencil code << 25)
constexpr uint32_t kIndexMask = (1u << kCodeShift) - 1u;

// Stencil code of a neighbour: offsets o in -2..2 per dimension,
// code = (ox+2) + 5 (oy+2) + 25 (oz+2).
__device__ __forceinline__ uint32_t make_code(int ox, int oy, int oz) {
  return (uint32_t)((ox + 2) + 5 * (oy + 2) + 25 * (oz + 2));
}

struct Offsets {
  int ox, oy, oz;
};
__device__ __forceinline__ Offsets decode_code(uint32_t code) {
  Offsets o;
  o.ox = (int)(code % 5u) - 2;
  o.oy = (int)((code / 5u) % 5u) - 2;
  o.oz = (int)(code / 25u) - 2;
  return o;
}

// FP64 lists store the neighbour's periodic image instead of its stencil
// offset: bits 25-26, 27-28 and 29-30 hold, per dimension, the image
// shift of x_i - x_j in box lengths as a 2-bit signed field (+1 for a
// virtual cell below 0, -1 for one at or above nm, else 0); bit 31 flags
// a colloid boundary particle.  The FP32 path needs the offsets
// (cell-relative positions) and keeps the codes.
struct Images {
  int sx, sy, sz;
};
// Bit 31 of an FP64 entry: the neighbour is a colloid boundary particle
// (boxes with colloids), so the pair body needs no species gather for the
// fluid-fluid pairs.
constexpr uint32_t kBoundaryBit = 0x80000000u;
__device__ __forceinline__ int image_class(int v, int nm) { return v < 0 ? 1 : (v >= nm ? -1 : 0); }
__device__ __forceinline__ uint32_t image_field(int v, int nm, int dim) {
  return ((uint32_t)image_class(v, nm) & 3u) << (kCodeShift + 2 * dim);
}
__device__ __forceinline__ Images decode_images(uint32_t ent) {
  Images m;
  m.sx = (int)(ent << 5) >> 30;
  m.sy = (int)(ent << 3) >> 30;
  m.sz = (int)(ent << 1) >> 30;
  return m;
}

// The cell-relative position of an xa record without its cell index: a
// 12-byte gather instead of 16.
__device__ __forceinline__ float4 load_xyz(const float4* __restrict__ rec) {
  const float* f = reinterpret_cast<const float*>(rec);
  return make_float4(f[0], f[1], f[2], 0.f);
}

// Geometry of the replica a chunk belongs to (uniform across the wave).
struct Geo {
  int nm0, nm1, nm2;    // sort-grid cells per dimension
  int cell_base, row_base;
  double L0, L1, L2;    // edge lengths
  double csd0;          // FP64 cell edge along x
  double half2;         // squared half of the shortest edge, a rounding margin less
  float cs0, cs1, cs2;  // FP32 cell edges
  float u0h, u1h, u2h, u0l, u1l, u2l;  // units of the fixed-point positions
};

// Lees-Edwards view of a lane (P.le_g >= 0).  Rows across the upper face
// (sigma 0) see the neighbours' upper copies, shifted along x by the shear
// length S_up = (v_upper - v_lower) t; rows across the lower face (sigma 1)
// by S_down = -S_up.  In the frame shifted by sp = MODULO(S, Lx) the lane
// sits in cell wc, dxf = (cx - wc) cs - sp is its FP32 offset from its own
// cell corner in that frame, and wmin / wmax bound wc over the wave.
// Per-lane Lees-Edwards frame of the two sheared faces (sigma 0: across
// the upper face, 1: across the lower face): x shift S' of the images, the
// window centre, the FP32 x offset of the sheared frame, and the wave's
// window range.  Named members with select accessors: an array indexed by
// the run-time sigma would be placed in scratch memory.
struct LeLane {
  double t;             // time of the shear length
  double sp0, sp1;
  int wc0, wc1;
  float dxf0, dxf1;
  int wmin0, wmin1, wmax0, wmax1;
  __device__ __forceinline__ double sp(int s) const { return s == 0 ? sp0 : sp1; }
  __device__ __forceinline__ int wc(int s) const { return s == 0 ? wc0 : wc1; }
  __device__ __forceinline__ float dxf(int s) const { return s == 0 ? dxf0 : dxf1; }
  __device__ __forceinline__ int wmin(int s) const { return s == 0 ? wmin0 : wmin1; }
  __device__ __forceinline__ int wmax(int s) const { return s == 0 ? wmax0 : wmax1; }
};

// Per-lane context of the home particle.
struct Home {
  int i;                // own index (valid for active lanes)
  int ii;               // a safe index for every lane
  bool active;
  int cx, cy, cz;       // own cell (replica-local)
  float4 a;             // FP32 position relative to the own cell corner
  double x0, x1, x2;    // FP64 position
  Geo G;
  LeLane le;
};

// Lees-Edwards sign of the stencil row at offsets (dy, dz): 0 across the
// upper face of the shearing dimension, 1 across the lower face, -1 none
__device__ __forceinline__ int le_sigma(const DevParams& P, const Home& h, int dy, int dz) {
  if (P.le_g == 1) {
    const int c = h.cy + dy;
    return c >= h.G.nm1 ? 0 : (c < 0 ? 1 : -1);
  }
  if (P.le_g == 2) {
    const int c = h.cz + dz;
    return c >= h.G.nm2 ? 0 : (c < 0 ? 1 : -1);
  }
  return -1;
}
// The same sign from a listed neighbour's images: the image below the
// upper face (shift -1) is the upper copy.
__device__ __forceinline__ int le_sigma(const DevParams& P, const Images& m) {
  const int c = P.le_g == 1 ? m.sy : (P.le_g == 2 ? m.sz : 0);
  return c < 0 ? 0 : (c > 0 ? 1 : -1);
}

// Image modes of a neighbour at offsets o from the home cell.
struct Modes {
  int m0, m1, m2;
};
// Exact FP64 difference and squared distance for a pair.
template <int DIM>
__device__ __forceinline__ double exact_d2(const DevParams& P, const double* __restrict__ x, int j,
                                           const Home& h, const Modes& m, double& d0, double& d1,
                                           double& d2) {
  const int64_t n = P.n;
  d0 = image_diff(h.x0, x[j], h.G.L0, m.m0);
  d1 = image_diff(h.x1, x[n + j], h.G.L1, m.m1);
  d2 = DIM == 3 ? image_diff(h.x2, x[2 * n + j], h.G.L2, m.m2) : 0.0;
  return DIM == 3 ? dist2_exact(d0, d1, d2) : dist2_exact2(d0, d1);
}

// Exact FP64 squared distance of a pair with the image chosen from the
// positions (image_diff_pos): the reference's formula and convention
// without the cell classes, so it holds between sorts (Verlet lists),
// after either particle crossed a periodic face.
template <int DIM>
__device__ __forceinline__ double exact_d2_pos(const DevParams& P, const Home& h, double xj0,
                                               double xj1, double xj2, double& d0, double& d1,
                                               double& d2) {
  d0 = image_diff_pos(h.x0, xj0, h.G.L0, P.symmetry);
  d1 = image_diff_pos(h.x1, xj1, h.G.L1, P.symmetry);
  d2 = DIM == 3 ? image_diff_pos(h.x2, xj2, h.G.L2, P.symmetry) : 0.0;
  return DIM == 3 ? dist2_exact(d0, d1, d2) : dist2_exact2(d0, d1);
}

// The Verlet lists' decision: the exact squared distance on the current
// positions with the image taken from them.  In a box with sheared faces a
// pair whose coordinates along the faces' normal differ by more than half
// the box meets across a face, and j's copy there is the one the candidate
// scan sees: sigma 0, the copy above the upper face, or 1, below the lower
// one (returned in sg; -1 when no sheared face lies between them), with the
// formula and roundings of exact_d2_le.
template <int DIM>
__device__ __forceinline__ double exact_d2_image(const DevParams& P, const Home& h, double xj0,
                                                  double xj1, double xj2, double& d0,
                                                  double& d1, double& d2, int& sg) {
  sg = -1;
  if (P.le_g >= 0) {
    const bool gy = P.le_g == 1;
    const double raw = gy ? h.x1 - xj1 : h.x2 - xj2;
    const double Lg = gy ? h.G.L1 : h.G.L2;
    sg = raw > 0.5 * Lg ? 0 : (raw < -0.5 * Lg ? 1 : -1);
  }
  if (sg < 0) return exact_d2_pos<DIM>(P, h, xj0, xj1, xj2, d0, d1, d2);
  const double L0 = h.G.L0;
  const double su = (P.le_vhi - P.le_vlo) * h.le.t, sd = (P.le_vlo - P.le_vhi) * h.le.t;
  double xi = h.x0, xj = xj0;
  if (sg == 0)
    xj = f_modulo(xj + su, L0);
  else if (P.symmetry)
    xi = f_modulo(xi + su, L0);
  else
    xj = f_modulo(xj + sd, L0);
  const double rx = xi - xj;
  const int mx = rx > 0.5 * L0 ? 1 : (rx < -0.5 * L0 ? (P.symmetry ? 2 : 3) : 0);
  const int mg = sg == 0 ? 1 : (P.symmetry ? 2 : 3);
  d0 = image_diff(xi, xj, L0, mx);
  if (P.le_g == 1) {
    d1 = image_diff(h.x1, xj1, h.G.L1, mg);
    d2 = DIM == 3 ? image_diff_pos(h.x2, xj2, h.G.L2, P.symmetry) : 0.0;
  } else {
    d1 = image_diff_pos(h.x1, xj1, h.G.L1, P.symmetry);
    d2 = image_diff(h.x2, xj2, h.G.L2, mg);
  }
  return DIM == 3 ? dist2_exact(d0, d1, d2) : dist2_exact2(d0, d1);
}

// The plain coordinate differences of a pair and their squared distance as
// the reference rounds it.  When that distance is at most half the shortest
// edge (G.half2), no coordinate differs by more than half its edge and no
// face lies between the two: exact_d2_image would return the same bits.
// Only the few pairs across a face then take its selects, about 36 of the
// 172 vector instructions an FP64 force pair took with them.
template <int DIM>
__device__ __forceinline__ double plain_d2(const Home& h, double xj0, double xj1, double xj2,
                                           double& d0, double& d1, double& d2) {
  d0 = h.x0 - xj0;
  d1 = h.x1 - xj1;
  d2 = DIM == 3 ? h.x2 - xj2 : 0.0;
  return DIM == 3 ? dist2_exact(d0, d1, d2) : dist2_exact2(d0, d1);
}

template <int DIM>
__device__ __forceinline__ double exact_d2_verlet(const DevParams& P, const Home& h, double xj0,
                                                  double xj1, double xj2, double& d0,
                                                  double& d1, double& d2, int& sg) {
  sg = -1;
  double r2 = plain_d2<DIM>(h, xj0, xj1, xj2, d0, d1, d2);
  if (!(r2 <= h.G.half2)) r2 = exact_d2_image<DIM>(P, h, xj0, xj1, xj2, d0, d1, d2, sg);
  return r2;
}

// FP32 squared distance, rounded as the candidate scan rounds it, so the
// in / out decisions of the density and force passes coincide
__device__ __forceinline__ float mixed_s2(float d0, float d1, float d2) {
  return fmaf(d2, d2, fmaf(d1, d1, d0 * d0));
}

// FP32 separation of fixed-point positions: the integer difference is the
// nearest image's, and the two-part unit keeps its scale exact to 2^-48 (a
// rounded scale would shift every distance, and the pressure with them).
template <int DIM>
__device__ __forceinline__ void fixed_diff(const Home& h, const uint4& a, const uint4& b, float& d0,
                                           float& d1, float& d2) {
  const float c0 = (float)(int32_t)(a.x - b.x), c1 = (float)(int32_t)(a.y - b.y);
  d0 = fmaf(c0, h.G.u0h, c0 * h.G.u0l);
  d1 = fmaf(c1, h.G.u1h, c1 * h.G.u1l);
  if (DIM == 3) {
    const float c2 = (float)(int32_t)(a.z - b.z);
    d2 = fmaf(c2, h.G.u2h, c2 * h.G.u2l);
  } else {
    d2 = 0.f;
  }
}

// FP32 separation from cell-relative positions and the stencil offsets.
template <int DIM>
__device__ __forceinline__ void rel_diff(const DevParams& P, const Home& h, const float4& q,
                                         const Offsets& o, float& d0, float& d1, float& d2) {
  float ax = h.a.x;
  if (P.le_g >= 0) {
    // across a Lees-Edwards face ox counts from the sheared window centre
    const int sg = le_sigma(P, h, o.oy, o.oz);
    if (sg >= 0) ax = ax + h.le.dxf(sg);
  }
  d0 = ax - (q.x + (float)o.ox * h.G.cs0);
  d1 = h.a.y - (q.y + (float)o.oy * h.G.cs1);
  d2 = DIM == 3 ? h.a.z - (q.z + (float)o.oz * h.G.cs2) : 0.f;
}

// The chunk of the sort grid this wavefront works on; false when the wave
// has none (the launch covers an upper bound of chunks).
struct Chunk {
  int c;                // chunk index
  int row;              // global row; replica-local row = cy + nm1 * cz
  int p0, p1;           // particles [p0, p1)
  int xmin, xmax;       // x range of the home cells
  Geo G;
};

// Chunk slots of the pair launches: an upper bound of the chunks (one
// partial chunk per row plus n / 64 full ones), rounded up to a multiple of
// the eight XCDs.
__host__ __device__ inline int chunk_slots(const DevParams& P) {
  const int m = (P.n + kWave - 1) / kWave + P.nrows;
  return (m + 7) / 8 * 8;
}

// Workgroups are handed to the eight XCDs round-robin.  With xcd_order,
// slot b takes chunk (b % 8) ceil(chunks / 8) + b / 8, i.e. each XCD
// works through a contiguous eighth of the chunk sequence and its L2 serves
// a compact slab of space; otherwise chunk b.  The slots, a multiple of 8
// (chunk_slots), are at least the number of chunks; a workgroup takes slot
// blockIdx.x, or every gridDim.x-th slot on the reduced grid of a rescan.
__device__ __forceinline__ bool load_chunk(const DevParams& P, const DeviceState& S, Chunk& ch,
                                           int b) {
  const int total = S.row_chunk_off[P.nrows];
  int c = b;
  if (P.xcd_order) {
    const int per = (total + 7) >> 3;
    c = (b & 7) * per + (b >> 3);
    if ((b >> 3) >= per) return false;
  }
  if (c >= total) return false;
  ch.c = c;
  ch.row = S.chunk_row[c];
  const int k = c - S.row_chunk_off[ch.row];
  const RepGeom& g = S.geo[S.row_rep[ch.row]];
  ch.G.nm0 = g.nm[0];
  ch.G.nm1 = g.nm[1];
  ch.G.nm2 = g.nm[2];
  ch.G.cell_base = g.cell_base;
  ch.G.row_base = g.row_base;
  ch.G.L0 = g.L[0];
  ch.G.L1 = g.L[1];
  ch.G.L2 = g.L[2];
  ch.G.csd0 = g.cs[0];
  const double lmin = fmin(fmin(g.L[0], g.L[1]), P.dim == 3 ? g.L[2] : g.L[1]);
  ch.G.half2 = 0.25 * lmin * lmin * (1.0 - 1e-13);
  ch.G.u0h = g.fhi[0];
  ch.G.u1h = g.fhi[1];
  ch.G.u2h = g.fhi[2];
  ch.G.u0l = g.flo[0];
  ch.G.u1l = g.flo[1];
  ch.G.u2l = g.flo[2];
  ch.G.cs0 = g.csf[0];
  ch.G.cs1 = g.csf[1];
  ch.G.cs2 = g.csf[2];
  const int c0 = S.row_cell[ch.row];
  const int rs = S.start[c0];
  const int re = S.start[c0 + ch.G.nm0];
  ch.p0 = rs + kWave * k;
  ch.p1 = min(ch.p0 + kWave, re);
  ch.xmin = (S.key_sorted[ch.p0] - ch.G.cell_base) % ch.G.nm0;
  ch.xmax = (S.key_sorted[ch.p1 - 1] - ch.G.cell_base) % ch.G.nm0;
  return true;
}

// Neighbour list block of a chunk of m particles: list_cap / 8 groups, each m
// lanes x 8 entries; a lane's group g holds its entries 8g .. 8g+7.  Verlet
// lists store them as (0, 4), (1, 5), (2, 6), (3, 7): four lanes walk a
// particle's list, lane s takes the entries s and s + 4 of a group in one
// 8-byte load, and a wave's 64 loads are contiguous.  The blocks follow the
// particles without padding (list_entries: the last lanes of the last block
// may read, not use, entries past it).
__device__ __forceinline__ uint32_t* list_block(const DevParams& P, uint32_t* list, const Chunk& ch) {
  return list + (int64_t)ch.p0 * P.list_cap;
}
__device__ __forceinline__ int64_t group_offset(const Chunk& ch, int q, int lane) {
  return ((q >> 3) * (ch.p1 - ch.p0) + lane) * 8;
}

template <int DIM>
__device__ __forceinline__ Home load_home(const DevParams& P, const DeviceState& S,
                                          const Chunk& ch) {
  Home h;
  const int lane = threadIdx.x;
  h.i = ch.p0 + lane;
  h.active = h.i < ch.p1;
  h.ii = h.active ? h.i : ch.p0;
  const int64_t n = P.n;
  h.G = ch.G;
  h.cx = (S.key_sorted[h.ii] - ch.G.cell_base) % ch.G.nm0;
  const int lr = ch.row - ch.G.row_base;
  h.cy = lr % ch.G.nm1;
  h.cz = lr / ch.G.nm1;
  h.a = S.xa[h.ii];
  h.x0 = S.x[h.ii];
  h.x1 = S.x[n + h.ii];
  h.x2 = DIM == 3 ? S.x[2 * n + h.ii] : 0.0;
  if (P.le_g >= 0) {
    // boxes with Lees-Edwards faces start at 0 (the reference's MODULO)
    h.le.t = S.time_dev[1];
    const double cs = ch.G.csd0;
#pragma unroll
    for (int sg = 0; sg < 2; ++sg) {
      const double sl = sg == 0 ? (P.le_vhi - P.le_vlo) * h.le.t : (P.le_vlo - P.le_vhi) * h.le.t;
      const double sp = f_modulo(sl, ch.G.L0);
      // Verlet lists keep the build's cells, and the FP32 position goes on
      // from the build cell unwrapped: the window centre is taken in that
      // frame, so a lane that crossed an x face since stays with its wave
      const double xw = P.verlet ? (double)h.cx * cs + (double)h.a.x : h.x0;
      const int wc = window_cell(xw, h.cx, cs, sp);
      const float dxf = (float)((double)(h.cx - wc) * cs - sp);
      int mn = h.active ? wc : INT_MAX, mx = h.active ? wc : INT_MIN;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        mn = min(mn, __shfl_xor(mn, off));
        mx = max(mx, __shfl_xor(mx, off));
      }
      if (sg == 0) {
        h.le.sp0 = sp;
        h.le.wc0 = wc;
        h.le.dxf0 = dxf;
        h.le.wmin0 = mn;
        h.le.wmax0 = mx;
      } else {
        h.le.sp1 = sp;
        h.le.wc1 = wc;
        h.le.dxf1 = dxf;
        h.le.wmin1 = mn;
        h.le.wmax1 = mx;
      }
    }
  }
  return h;
}

// ---------------------------------------------------------------------
// stencil rows of a chunk
// ---------------------------------------------------------------------
// One stencil row (dy, dz) of a chunk covers the virtual cells
// [vlo, vhi] of the target row of cells: virtual cell v is physical cell
// v - m nm0 seen through m periodic x faces.  Lanes look at the five cells
// around their own (home cell, or the Lees-Edwards window centre), so the
// range is [xmin - 2, xmax + 2] (or the window centres' extremes +-2) and
// splits into at most three pieces of one period each, contiguous in
// memory: piece k spans virtual [a_k, a_k+1) of period m0 + k.  Sequence
// index t runs over the pieces in that order.
struct RowPieces {
  int rb;                 // first cell of the target row
  int my, mz;             // image modes of the row in y and z
  int sigma;              // Lees-Edwards sign of the row (-1 none)
  int vlo, a1, a2, aend;  // piece bounds in virtual cells
  int m0;                 // period of piece 0
  int g0, len0, g1, len1, g2, len2;
  int tot;
};

__device__ __forceinline__ int floor_div(int a, int b) {
  return a >= 0 ? a / b : -((-a + b - 1) / b);
}

template <int DIM>
__device__ __forceinline__ RowPieces row_pieces(const DevParams& P, const DeviceState& S,
                                                const Chunk& ch, const Home& h, int row) {
  RowPieces rp;
  const int nm0 = h.G.nm0;
  const int32_t* __restrict__ start = S.start;
  const int dy = row % 5 - 2, dz = DIM == 3 ? row / 5 - 2 : 0;
  rp.mz = 0;
  const int ny = wrap_cell(h.cy + dy, h.G.nm1, P.symmetry, rp.my);
  const int nz = DIM == 3 ? wrap_cell(h.cz + dz, h.G.nm2, P.symmetry, rp.mz) : 0;
  rp.rb = h.G.cell_base + nm0 * (ny + h.G.nm1 * nz);
  rp.sigma = P.le_g >= 0 ? le_sigma(P, h, dy, dz) : -1;
  int vhi;
  if (rp.sigma < 0) {
    rp.vlo = ch.xmin - 2;
    vhi = ch.xmax + 2;
  } else {
    rp.vlo = h.le.wmin(rp.sigma) - 2;
    vhi = h.le.wmax(rp.sigma) + 2;
  }
  rp.aend = vhi + 1;
  rp.m0 = floor_div(rp.vlo, nm0);
  rp.a1 = min(rp.aend, (rp.m0 + 1) * nm0);
  rp.a2 = min(rp.aend, (rp.m0 + 2) * nm0);
  const int b0 = rp.m0 * nm0, b1 = b0 + nm0, b2 = b1 + nm0;
  rp.g0 = start[rp.rb + rp.vlo - b0];
  rp.len0 = start[rp.rb + rp.a1 - b0] - rp.g0;
  rp.g1 = rp.a2 > rp.a1 ? start[rp.rb + rp.a1 - b1] : rp.g0;
  rp.len1 = rp.a2 > rp.a1 ? start[rp.rb + rp.a2 - b1] - rp.g1 : 0;
  rp.g2 = rp.aend > rp.a2 ? start[rp.rb + rp.a2 - b2] : rp.g0;
  rp.len2 = rp.aend > rp.a2 ? start[rp.rb + rp.aend - b2] - rp.g2 : 0;
  rp.tot = rp.len0 + rp.len1 + rp.len2;
  return rp;
}

// sequence index of the first particle of virtual cell v (v in [vlo, aend])
__device__ __forceinline__ int seq_of(const RowPieces& rp, const int32_t* __restrict__ start,
                                      int nm0, int v) {
  if (v >= rp.aend) return rp.tot;
  const int b0 = rp.m0 * nm0;
  if (v < rp.a1) return start[rp.rb + v - b0] - rp.g0;
  if (v < rp.a2) return rp.len0 + (start[rp.rb + v - b0 - nm0] - rp.g1);
  return rp.len0 + rp.len1 + (start[rp.rb + v - b0 - 2 * nm0] - rp.g2);
}

// particle index of sequence position t
__device__ __forceinline__ int seq_particle(const RowPieces& rp, int t) {
  return t < rp.len0 ? rp.g0 + t
                     : (t < rp.len0 + rp.len1 ? rp.g1 + (t - rp.len0) : rp.g2 + (t - rp.len0 - rp.len1));
}

// Exact FP64 squared distance of a pair across a Lees-Edwards face, as the
// reference forms it from its images (ppm_bcdef_le_y.inc, then the
// periodic cascade): the shifted copy is MODULO(x + shear_length, Lx)
// along x (j's upper copy for sigma 0; for sigma 1 i's upper copy with
// symmetry, j's lower copy without), whose periodic image nearest the
// other particle is the one inside the cut-off.
template <int DIM>
__device__ __forceinline__ double exact_d2_le(const DevParams& P, const double* __restrict__ x,
                                              int j, const Home& h, int sigma, int my, int mz) {
  const int64_t n = P.n;
  const double L0 = h.G.L0;
  const double su = (P.le_vhi - P.le_vlo) * h.le.t, sd = (P.le_vlo - P.le_vhi) * h.le.t;
  double xi = h.x0, xj = x[j];
  if (sigma == 0)
    xj = f_modulo(xj + su, L0);
  else if (P.symmetry)
    xi = f_modulo(xi + su, L0);
  else
    xj = f_modulo(xj + sd, L0);
  const double raw = xi - xj;
  const int mx = raw > 0.5 * L0 ? 1 : (raw < -0.5 * L0 ? (P.symmetry ? 2 : 3) : 0);
  const int mg = sigma == 0 ? 1 : (P.symmetry ? 2 : 3);
  const double d0 = image_diff(xi, xj, L0, mx);
  const double d1 = image_diff(h.x1, x[n + j], h.G.L1, P.le_g == 1 ? mg : my);
  if (DIM == 2) return dist2_exact2(d0, d1);
  const double d2 = image_diff(h.x2, x[2 * n + j], h.G.L2, P.le_g == 2 ? mg : mz);
  return dist2_exact(d0, d1, d2);
}

// ---------------------------------------------------------------------
// the staged scan
// ---------------------------------------------------------------------
// Candidate scan over the stencil rows of a chunk; returns the number of
// accepted neighbours.
// SKIN (Verlet lists): accept every candidate within rc + skin (FP32, with
// the band's margin); the policy's body takes the in / out decision.
template <int DIM, class Pol, int TILE = kTile, int BUF = kBuf, bool SKIN = false>
__device__ __forceinline__ int staged_scan(const DevParams& P, const DeviceState& S,
                                           const Chunk& ch, const Home& h, Pol& pol,
                                           float4* __restrict__ tile, uint32_t* __restrict__ buf,
                                           int& rechecks, uint32_t* __restrict__ list) {
  const int lane = threadIdx.x;
  const int nm0 = h.G.nm0;
  const int32_t* __restrict__ start = S.start;
  const int low_mode = P.symmetry ? 2 : 3;
  // the boundary flag of the lane's own record (FP64 entries with colloids)
  const uint32_t self_flag = (Pol::kImages && P.ncoll && S.sid[h.ii] != 0) ? kBoundaryBit : 0u;
  int cnt = 0, stored = 0;
  // buf holds cnt entries of this lane, the first ev of them evaluated
  // already; entries reach the list block in whole groups of 8
  int ev = 0;
  uint32_t* __restrict__ blk = list ? list_block(P, list, ch) : nullptr;
  auto flush = [&](bool final) {
    if constexpr (Pol::kBatched) {
      // Pol::kBatch entries at a time: the policy issues all their gathers
      // before it evaluates the first pair (slots past cnt read the lane's
      // own particle and add nothing)
      constexpr int NB = Pol::kBatch;
      for (int q = ev; __ballot(q < cnt) != 0ull; q += NB) {
        uint32_t e[NB];
        bool ok[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          ok[k] = q + k < cnt;
          e[k] = ok[k] ? buf[(q + k) * kWave + lane] : (uint32_t)h.ii;
        }
        pol.body_batch(e, ok);
      }
    } else {
      for (int q = ev; __ballot(q < cnt) != 0ull; ++q) {
        if (q < cnt) {
          pol.body(buf[q * kWave + lane]);
        }
      }
    }
    const int w = final ? cnt : (cnt & ~7);
    if (blk) {
      for (int q = 0; __ballot(q < w) != 0ull; q += 8) {
        if (q < w && stored + q + 8 <= P.list_cap) {
          // (SKIN: Verlet lists, entries paired for the four-lane walk)
          uint4 lo, hi;
          lo.x = buf[(q + 0) * kWave + lane];
          lo.y = buf[(q + (SKIN ? 4 : 1)) * kWave + lane];
          lo.z = buf[(q + (SKIN ? 1 : 2)) * kWave + lane];
          lo.w = buf[(q + (SKIN ? 5 : 3)) * kWave + lane];
          hi.x = buf[(q + (SKIN ? 2 : 4)) * kWave + lane];
          hi.y = buf[(q + (SKIN ? 6 : 5)) * kWave + lane];
          hi.z = buf[(q + (SKIN ? 3 : 6)) * kWave + lane];
          hi.w = buf[(q + 7) * kWave + lane];
          uint4* dst = reinterpret_cast<uint4*>(blk + group_offset(ch, stored + q, lane));
          dst[0] = lo;
          dst[1] = hi;
        }
      }
    }
    stored += w;
    // keep the unwritten tail (fewer than 8 entries) at the front
    const int rem = cnt - w;
    for (int r = 0; r < rem; ++r) buf[r * kWave + lane] = buf[(w + r) * kWave + lane];
    cnt = rem;
    ev = rem;
  };
  const int nrow = DIM == 3 ? 25 : 5;
#pragma unroll 1
  for (int row = 0; row < nrow; ++row) {
    const int dy = row % 5 - 2, dz = DIM == 3 ? row / 5 - 2 : 0;
    const RowPieces rp = row_pieces<DIM>(P, S, ch, h, row);
    const int my = rp.my, mz = rp.mz;
    const int tot = rp.tot;
    const int v_lo = rp.vlo;
    // Positions in the tile are relative to the corner of virtual cell
    // v_lo in x (and to the candidate's own cell in y, z).  With stencil
    // codes the tile's .w holds the list entry with the virtual cell (mod
    // 128) in place of the code, so that entry + kadd is the entry with
    // the code (the offset from the lane's window centre); with images it
    // holds the entry with the x image, and the row adds the y and z ones.
    // Across a Lees-Edwards face the window centre and the lane's x come
    // from the sheared frame.
    const bool le_row = rp.sigma >= 0;
    const int wc = le_row ? h.le.wc(rp.sigma) : h.cx;
    const int crel = wc - v_lo;
    const float ax = (le_row ? h.a.x + h.le.dxf(rp.sigma) : h.a.x) + (float)crel * h.G.cs0;
    // the lane's own copy: same particle, own virtual cell (x image 0)
    const uint32_t self_w =
        le_row ? 0xFFFFFFFFu
               : (Pol::kImages ? ((uint32_t)h.ii | self_flag)
                               : ((uint32_t)h.ii | ((uint32_t)crel << kCodeShift)));
    // this lane's window: virtual cells wc-2 .. wc+2 as a range of the
    // row sequence
    int tb = 0, te = 0;
    if (h.active) {
      tb = seq_of(rp, start, nm0, wc - 2);
      te = seq_of(rp, start, nm0, wc + 3);
    }
    const float ay = h.a.y - (float)dy * h.G.cs1;
    const float az = DIM == 3 ? h.a.z - (float)dz * h.G.cs2 : 0.f;
    const uint32_t kadd =
        Pol::kImages
            ? image_field(h.cy + dy, h.G.nm1, 1) | (DIM == 3 ? image_field(h.cz + dz, h.G.nm2, 2) : 0u)
            : (uint32_t)(2 - crel + 5 * (dy + 2) + 25 * (dz + 2)) << kCodeShift;
    // the row in batches of at most TILE records (one batch in practice)
    for (int base = 0; base < tot; base += TILE) {
      const int bend = min(tot, base + TILE);
      for (int t = base + lane; t < bend; t += kWave) {
        const int piece = t < rp.len0 ? 0 : (t < rp.len0 + rp.len1 ? 1 : 2);
        const int g = seq_particle(rp, t);
        const float4 q = S.xa[g];
        const int v = __float_as_int(q.w) + (rp.m0 + piece) * nm0;
        const int vrel = v - v_lo;
        uint32_t code = Pol::kImages ? image_field(v, nm0, 0) : (uint32_t)vrel << kCodeShift;
        if (Pol::kImages && P.ncoll && S.sid[g] != 0) code |= kBoundaryBit;
        tile[t - base] = make_float4(fmaf((float)vrel, h.G.cs0, q.x), q.y, q.z,
                                     __uint_as_float((uint32_t)g | code));
      }
      __syncthreads();
      const int lb = max(tb, base) - base, le = min(te, bend) - base;
      for (int t = lb; __ballot(t < le) != 0ull; t += 2) {
        if (__ballot(cnt > BUF - 2) != 0ull) flush(false);
        // records t and t + 1 from one clamped base (the tile holds TILE + 1
        // records; a clamped base only serves lanes past their window)
        const float4* __restrict__ tp = tile + min(t, TILE - 1);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int tt = t + u;
          const bool live = tt < le;
          const float4 q = tp[u];
          const uint32_t wv = __float_as_uint(q.w);
          const float d0 = ax - q.x;
          const float d1 = ay - q.y;
          float s2 = fmaf(d1, d1, d0 * d0);
          if (DIM == 3) {
            const float d2 = az - q.z;
            s2 = fmaf(d2, d2, s2);
          }
          const bool ok = live && wv != self_w;
          const uint32_t ent = wv + kadd;
          const bool below_lo = SKIN ? s2 < P.skin2_hi_f32 : s2 < P.cut2_lo_f32;
          const bool below_hi = SKIN ? below_lo : s2 < P.cut2_hi_f32;
          bool in = below_lo;
          if (!SKIN && ok && below_hi && !below_lo) {
            // FP64 re-decision with the reference's image convention
            ++rechecks;
            const int j = (int)(ent & kIndexMask);
            if (le_row) {
              in = exact_d2_le<DIM>(P, S.x, j, h, rp.sigma, my, mz) < P.cut2;
            } else {
              const int cls = Pol::kImages ? decode_images(ent).sx
                                           : image_class(h.cx + decode_code(ent >> kCodeShift).ox, nm0);
              Modes m;
              m.m0 = cls > 0 ? low_mode : (cls < 0 ? 1 : 0);
              m.m1 = my;
              m.m2 = mz;
              double e0, e1, e2;
              in = exact_d2<DIM>(P, S.x, j, h, m, e0, e1, e2) < P.cut2;
            }
          }
          if (ok && in) {
            buf[cnt * kWave + lane] = ent;
            ++cnt;
          }
        }
      }
      __syncthreads();
    }
  }
  flush(true);
  return stored;
}

// The scan of a list build: the entries of staged_scan with SKIN, in the same
// order, stored and not evaluated (the walk of the same step does that).
// LANES: with 1 a wave takes the chunk, a lane per particle.  With 4 it takes 16
// of the chunk's particles (ch is cut to them), and four lanes test four
// candidates of a particle at a time; a ballot gives each its place, so the
// entries stand in the same order.  stride, own: particles of the chunk and the
// lane's particle among them (the layout of the lists).
//
// A wave per chunk leaves small boxes a chain of latencies, so nothing waits
// within a row: lane r looks up stencil row r before the first one starts, and
// a row's records and window bounds load while the row before is scanned.
// A build without its sums takes 83 us instead of 185 in a 32^3 box (mixed
// precision) and 0.97 ms instead of 2.2 in the 128^3 one (1.53 with the
// registers of two waves per SIMD); the walk adds 22 us and 0.58 ms.
// tile holds TILE + kTilePad<LANES> records (the last ones only serve lanes
// past their window).
template <int LANES>
constexpr int kTilePad = LANES == 4 ? 7 : 3;
template <int DIM, bool IMAGES, int TILE, int BUF, int LANES = 1>
__device__ __forceinline__ int list_scan(const DevParams& P, const DeviceState& S,
                                         const Chunk& ch, const Home& h, int stride, int own,
                                         float4* __restrict__ tile, uint32_t* __restrict__ buf,
                                         uint32_t* __restrict__ blk) {
  constexpr int kRows = DIM == 3 ? 25 : 5;
  constexpr int kAhead = (TILE + kWave - 1) / kWave;  // records per lane of a row's first batch
  constexpr int kStep = 4;                            // candidates per lane and pass
  constexpr int kRing = (BUF + 7) / 8 * 8;            // rows of buf: a ring of whole groups
  static_assert((kRing & (kRing - 1)) == 0 && kRing >= 8 + kStep, "");
  const int lane = threadIdx.x;
  // four lanes per particle: buf holds kDeep entries of each of 16 particles
  constexpr int kDeep = 4 * kRing;
  const int part = lane >> 2, sub = lane & 3;
  // the waves of a workgroup share nothing here (one wave: LDS operations
  // complete in order)
  auto sync = [&]() {
    if constexpr (LANES == 1)
      __syncthreads();
    else
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  const int nm0 = h.G.nm0;
  const int32_t* __restrict__ start = S.start;
  const uint32_t self_flag = (IMAGES && P.ncoll && S.sid[h.ii] != 0) ? kBoundaryBit : 0u;
  const RowPieces mine = row_pieces<DIM>(P, S, ch, h, lane < kRows ? lane : kRows - 1);
  auto row_of = [&](int row) {
    RowPieces rp;
    auto get = [&](int v) { return __builtin_amdgcn_readlane(v, row); };
    rp.rb = get(mine.rb);
    rp.my = get(mine.my);
    rp.mz = get(mine.mz);
    rp.sigma = get(mine.sigma);
    rp.vlo = get(mine.vlo);
    rp.a1 = get(mine.a1);
    rp.a2 = get(mine.a2);
    rp.aend = get(mine.aend);
    rp.m0 = get(mine.m0);
    rp.g0 = get(mine.g0);
    rp.len0 = get(mine.len0);
    rp.g1 = get(mine.g1);
    rp.len1 = get(mine.len1);
    rp.g2 = get(mine.g2);
    rp.len2 = get(mine.len2);
    rp.tot = get(mine.tot);
    return rp;
  };
  // a record of the row's sequence with its entry, ready for the tile
  struct Rec {
    float4 q;
    int sid;
  };
  auto fetch = [&](const RowPieces& rp, int t) {
    const int g = seq_particle(rp, min(t, rp.tot - 1));
    Rec r;
    r.q = S.xa[g];
    r.sid = (IMAGES && P.ncoll) ? S.sid[g] : 0;
    return r;
  };
  auto place = [&](const RowPieces& rp, int t, const Rec& r, float4* __restrict__ to) {
    const int g = seq_particle(rp, t);
    const int piece = t < rp.len0 ? 0 : (t < rp.len0 + rp.len1 ? 1 : 2);
    const int v = __float_as_int(r.q.w) + (rp.m0 + piece) * nm0;
    const int vrel = v - rp.vlo;
    uint32_t code = IMAGES ? image_field(v, nm0, 0) : (uint32_t)vrel << kCodeShift;
    if (IMAGES && P.ncoll && r.sid != 0) code |= kBoundaryBit;
    *to = make_float4(fmaf((float)vrel, h.G.cs0, r.q.x), r.q.y, r.q.z,
                      __uint_as_float((uint32_t)g | code));
  };
  // the lane's entries so far, and those of them (whole groups of 8) in its
  // list; entry q waits in row q mod kRing of buf
  int cnt = 0, stored = 0;
  auto flush = [&](int least) {
    if constexpr (LANES == 4) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      while (__ballot(cnt - stored >= least) != 0ull) {
        if (cnt - stored >= least) {
          if (stored + 8 <= P.list_cap)
            *reinterpret_cast<uint2*>(blk + ((stored >> 3) * stride + own) * 8 + 2 * sub) =
                make_uint2(buf[((stored + sub) & (kDeep - 1)) * 16 + part],
                           buf[((stored + sub + 4) & (kDeep - 1)) * 16 + part]);
          stored += 8;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      return;
    }
    if (cnt - stored >= least) {
      if (stored + 8 <= P.list_cap) {
        const uint32_t* __restrict__ from = buf + (stored & (kRing - 1)) * kWave + lane;
        // (pairs for the four-lane walk)
        uint4 lo, hi;
        lo.x = from[0 * kWave];
        lo.y = from[4 * kWave];
        lo.z = from[1 * kWave];
        lo.w = from[5 * kWave];
        hi.x = from[2 * kWave];
        hi.y = from[6 * kWave];
        hi.z = from[3 * kWave];
        hi.w = from[7 * kWave];
        uint4* dst = reinterpret_cast<uint4*>(blk + ((stored >> 3) * stride + own) * 8);
        dst[0] = lo;
        dst[1] = hi;
      }
      stored += 8;
    }
  };
  // what a row needs, loaded while the row before is scanned
  RowPieces rp = row_of(0);
  Rec ahead[kAhead];
  int wc = 0, tb = 0, te = 0;
  auto prepare = [&]() {
    wc = rp.sigma >= 0 ? h.le.wc(rp.sigma) : h.cx;
    // this lane's window: virtual cells wc-2 .. wc+2 as a range of the row
    // sequence
    tb = te = 0;
    if (h.active) {
      tb = seq_of(rp, start, nm0, wc - 2);
      te = seq_of(rp, start, nm0, wc + 3);
    }
    if (rp.tot > 0) {
#pragma unroll
      for (int k = 0; k < kAhead; ++k) ahead[k] = fetch(rp, lane + k * kWave);
    }
  };
  prepare();
#pragma unroll 1
  for (int row = 0; row < kRows; ++row) {
    const RowPieces now = rp;
    const int wc_now = wc, tb_now = tb, te_now = te;
    const int dy = row % 5 - 2, dz = DIM == 3 ? row / 5 - 2 : 0;
    // Positions in the tile are relative to the corner of virtual cell vlo in
    // x and to the candidate's own cell in y and z (staged_scan).
    const bool le_row = now.sigma >= 0;
    const int crel = wc_now - now.vlo;
    const float ax = (le_row ? h.a.x + h.le.dxf(now.sigma) : h.a.x) + (float)crel * h.G.cs0;
    const uint32_t self_w =
        le_row ? 0xFFFFFFFFu
               : (IMAGES ? ((uint32_t)h.ii | self_flag)
                         : ((uint32_t)h.ii | ((uint32_t)crel << kCodeShift)));
    const float ay = h.a.y - (float)dy * h.G.cs1;
    const float az = DIM == 3 ? h.a.z - (float)dz * h.G.cs2 : 0.f;
    const uint32_t kadd =
        IMAGES
            ? image_field(h.cy + dy, h.G.nm1, 1) | (DIM == 3 ? image_field(h.cz + dz, h.G.nm2, 2) : 0u)
            : (uint32_t)(2 - crel + 5 * (dy + 2) + 25 * (dz + 2)) << kCodeShift;
    for (int base = 0; base < now.tot; base += TILE) {
      const int bend = min(now.tot, base + TILE);
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int t = base + lane + k * kWave;
        if (k * kWave + lane < TILE && t < bend) {
          if (base > 0) ahead[k] = fetch(now, t);
          place(now, t, ahead[k], tile + (t - base));
        }
      }
      sync();
      if (bend == now.tot && row + 1 < kRows) {
        rp = row_of(row + 1);
        prepare();
      }
      const int lb = max(tb_now, base) - base, le = min(te_now, bend) - base;
      if constexpr (LANES == 4) {
        for (int t = lb; __ballot(t < le) != 0ull; t += 8) {
          if (__ballot(cnt - stored > kDeep - 8) != 0ull) flush(8);
          const float4* __restrict__ tp = tile + min(t, TILE - 1) + sub;
          const float4 qq[2] = {tp[0], tp[4]};
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const float4 q = qq[u];
            const uint32_t wv = __float_as_uint(q.w);
            const float d0 = ax - q.x;
            const float d1 = ay - q.y;
            float s2 = fmaf(d1, d1, d0 * d0);
            if (DIM == 3) {
              const float d2 = az - q.z;
              s2 = fmaf(d2, d2, s2);
            }
            const bool in = t + 4 * u + sub < le && wv != self_w && s2 < P.skin2_hi_f32;
            const uint32_t four = (uint32_t)(__ballot(in) >> (lane & 60)) & 15u;
            if (in)
              buf[((cnt + __popc(four & ((1u << sub) - 1u))) & (kDeep - 1)) * 16 + part] = wv + kadd;
            cnt += __popc(four);
          }
        }
      } else
      for (int t = lb; __ballot(t < le) != 0ull; t += kStep) {
        if (__ballot(cnt - stored > kRing - kStep) != 0ull) flush(8);
        const float4* __restrict__ tp = tile + min(t, TILE - 1);
#pragma unroll
        for (int u = 0; u < kStep; ++u) {
          const float4 q = tp[u];
          const uint32_t wv = __float_as_uint(q.w);
          const float d0 = ax - q.x;
          const float d1 = ay - q.y;
          float s2 = fmaf(d1, d1, d0 * d0);
          if (DIM == 3) {
            const float d2 = az - q.z;
            s2 = fmaf(d2, d2, s2);
          }
          // (written in any case: the next entry overwrites it unless it counts)
          buf[(cnt & (kRing - 1)) * kWave + lane] = wv + kadd;
          cnt += (t + u < le && wv != self_w && s2 < P.skin2_hi_f32) ? 1 : 0;
        }
      }
      sync();
    }
    if (now.tot == 0 && row + 1 < kRows) {
      rp = row_of(row + 1);
      prepare();
    }
  }
  flush(8);
  flush(1);
  return cnt;
}

// FP32 terms summed in FP64 (each add rounds once, at FP64 precision)
struct WideF {
  double s = 0.0;
  __device__ __forceinline__ void add(float v) { s = s + (double)v; }
  __device__ __forceinline__ double value() const { return s; }
};

// compensated FP32 accumulator (Kahan)
struct KahanF {
  float s = 0.f, c = 0.f;
  __device__ __forceinline__ void add(float v) {
    float y = v - c;
    float t = s + y;
    c = (t - s) - y;
    s = t;
  }
  __device__ __forceinline__ double value() const { return (double)s - (double)c; }
};

// ---------------------------------------------------------------------
// K2: density + EOS
// ---------------------------------------------------------------------
// Velocity of a neighbour's Lees-Edwards copy relative to its own: + the
// face velocity jump across the upper face, - across the lower one
// (particles_set_boundary_ghost_velocity.F90:175-240).
__device__ __forceinline__ double le_dv(const DevParams& P, const Images& m) {
  if (P.le_g < 0) return 0.0;
  const int sg = le_sigma(P, m);
  return sg == 0 ? P.le_u : (sg == 1 ? -P.le_u : 0.0);
}
__device__ __forceinline__ float le_dvf(const DevParams& P, const Home& h, const Offsets& o) {
  if (P.le_g < 0) return 0.f;
  const int sg = le_sigma(P, h, o.oy, o.oz);
  return sg == 0 ? P.le_uf : (sg == 1 ? -P.le_uf : 0.f);
}

// FP64 separation of a listed pair: x_i - x_j plus the periodic image
// shift of the neighbour's virtual cell, s L with s in {-1, 0, 1} (the fma
// rounds once, as the sum with the shift does).  The in/out decision was
// taken with the reference's own formula; the value here differs from it
// by at most an ulp of the box length.
template <int DIM>
__device__ __forceinline__ double pair_d2(const DevParams& P, const Home& h, const Images& m,
                                          double xj0, double xj1, double xj2, double& d0,
                                          double& d1, double& d2) {
  d0 = fma((double)m.sx, h.G.L0, h.x0 - xj0);
  if (P.le_g >= 0) {
    // across a Lees-Edwards face: the sheared copy, nearest periodic image
    const int sg = le_sigma(P, m);
    if (sg >= 0) {
      // x_i - x_j - S' lies in (-2 Lx, Lx): nearest period
      const double raw = (h.x0 - xj0) - h.le.sp(sg);
      d0 = raw - h.G.L0 * rint(raw / h.G.L0);
    }
  }
  d1 = fma((double)m.sy, h.G.L1, h.x1 - xj1);
  d2 = DIM == 3 ? fma((double)m.sz, h.G.L2, h.x2 - xj2) : 0.0;
  return DIM == 3 ? fma(d2, d2, fma(d1, d1, d0 * d0)) : fma(d1, d1, d0 * d0);
}

// Element j of a device array, addressed as base + 32-bit byte offset (at
// most 2^25 elements of 16 bytes).
template <class T>
__device__ __forceinline__ T load_at(const T* base, uint32_t j) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) +
                                     (size_t)(j * (uint32_t)sizeof(T)));
}

// DECIDE (Verlet lists): the entries are candidates within rc + skin; the
// body takes the exact in / out decision on the current positions and
// counts the in-cut-off neighbours (nin) and the FP64 re-decisions.  The
// positions come as (x, y) from the record's first plane and z: two gathers
// per entry.
template <int DIM, bool DECIDE = false>
struct DensityF64 {
  const DevParams& P;
  const DeviceState& S;
  const Home& h;
  double acc;
  int nin = 0, rechecks = 0;
  static constexpr bool kImages = true;
  static constexpr bool kBatched = DECIDE;
  static constexpr int kBatch = 2;  // (larger ones cost the scan kernels registers)
  static constexpr int kTerms = 1;
  static constexpr int kWalk = 4;
  __device__ __forceinline__ void body(uint32_t ent) {
    const int j = (int)(ent & kIndexMask);
    const int64_t n = P.n;
    double d0, d1, d2;
    const double r2 = pair_d2<DIM>(P, h, decode_images(ent), S.x[j], S.x[n + j],
                                   DIM == 3 ? S.x[2 * n + j] : 0.0, d0, d1, d2);
    const double w = kernel_w(P, sqrt_pos(r2));
    acc = acc + (P.density_type == 1 ? S.m[j] * w : w);
  }
  // what a batch gathers, and the terms of its NB entries (0 outside the
  // cut-off and in empty slots)
  struct Rec {
    double2 a;
    double z;
  };
  __device__ __forceinline__ Rec gather(uint32_t ent) const {
    const uint32_t j = ent & kIndexMask;
    return {load_at(reinterpret_cast<const double2*>(S.rec64), j),
            DIM == 3 ? load_at(S.x + 2 * (int64_t)P.n, j) : 0.0};
  }
  template <int NB>
  __device__ __forceinline__ void terms(const uint32_t (&e)[NB], const bool (&ok)[NB],
                                        Rec (&r)[NB], double (&t)[NB][kTerms]) {
    // the reference's decision (pp_interaction.inc:37-46) on the current
    // positions; one branch of the wave for the batches with a pair across a
    // face
    double r2[NB];
    uint64_t far = 0;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      double d0, d1, d2;
      r2[k] = plain_d2<DIM>(h, r[k].a.x, r[k].a.y, r[k].z, d0, d1, d2);
      far |= __ballot(!(r2[k] <= h.G.half2));
    }
    if (__builtin_expect(far != 0, 0)) {
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        double d0, d1, d2;
        int sg;
        r2[k] = exact_d2_image<DIM>(P, h, r[k].a.x, r[k].a.y, r[k].z, d0, d1, d2, sg);
      }
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const bool use = ok[k] && r2[k] < P.cut2;
      nin += use ? 1 : 0;
      double w = kernel_w(P, sqrt_pos(r2[k]));
      if (P.density_type == 1) w = S.m[(int)(e[k] & kIndexMask)] * w;
      t[k][0] = use ? w : 0.0;
    }
  }
  template <int NB>
  __device__ __forceinline__ void body_batch(const uint32_t (&e)[NB], const bool (&ok)[NB]) {
    double t[NB][kTerms];
    Rec r[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) r[k] = gather(e[k]);
    terms(e, ok, r, t);
#pragma unroll
    for (int k = 0; k < NB; ++k) acc = acc + t[k][0];
  }
};

// Plain coordinate differences taken to the nearest image (one rounding, as
// pair_d2's; across a sheared face j's copy is moved by the shear length and
// jump is its extra x velocity).  False for a NaN separation, which an in /
// out decision leaves out: it goes outside the cut-off.
template <int DIM>
__device__ __forceinline__ bool nearest_image(const DevParams& P, const Home& h, double& d0,
                                              double& d1, double& d2, double& jump) {
  auto fold = [](double d, double L) {
    return d > 0.5 * L ? d - L : (d < -0.5 * L ? d + L : d);
  };
  if (P.le_g >= 0) {
    const double raw = P.le_g == 1 ? d1 : d2;
    const double Lg = P.le_g == 1 ? h.G.L1 : h.G.L2;
    const int sg = raw > 0.5 * Lg ? 0 : (raw < -0.5 * Lg ? 1 : -1);
    if (sg >= 0) {
      const double t = d0 - h.le.sp(sg);
      d0 = t - h.G.L0 * rint(t / h.G.L0);
      jump = sg == 0 ? P.le_u : -P.le_u;
    }
  }
  d0 = fold(d0, h.G.L0);
  d1 = fold(d1, h.G.L1);
  if (DIM == 3) d2 = fold(d2, h.G.L2);
  const double r2 = DIM == 3 ? dist2_exact(d0, d1, d2) : dist2_exact2(d0, d1);
  if (r2 <= h.G.half2) return true;
  d0 = 2.0 * P.cut_off;
  d1 = d2 = 0.0;
  return false;
}

// The in / out decision of a candidate from its FP32 squared distance: in
// below the band, out above it, inside it the reference's FP64 formula.
template <int DIM>
__device__ __forceinline__ bool mixed_inside(const DevParams& P, const DeviceState& S,
                                             const Home& h, int j, float s2, int& rechecks) {
  if (s2 < P.cut2_lo_f32) return true;
  if (!(s2 < P.cut2_hi_f32)) return false;
  ++rechecks;
  const int64_t n = P.n;
  double e0, e1, e2;
  return exact_d2_pos<DIM>(P, h, S.x[j], S.x[n + j], DIM == 3 ? S.x[2 * n + j] : 0.0, e0, e1,
                           e2) < P.cut2;
}

// Per-step lists: FP32 cell-relative positions, compensated FP32 sums.
template <int DIM>
struct DensityMixedStep {
  const DevParams& P;
  const DeviceState& S;
  const Home& h;
  KahanF acc;
  int nin = 0, rechecks = 0;
  static constexpr bool kImages = false;
  // in batches of eight (the 128^3 Tait box in mixed precision: 0.59 ms in
  // fours, 0.51 in eights, 0.55 in sixteens)
  static constexpr bool kBatched = true;
  static constexpr int kBatch = 8;
  template <int NB>
  __device__ __forceinline__ void body_batch(const uint32_t (&e)[NB], const bool (&ok)[NB]) {
    float4 q[NB];
    float mj[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int j = (int)(e[k] & kIndexMask);
      q[k] = load_xyz(S.xa + j);
      mj[k] = P.density_type == 1 ? (float)S.m[j] : 1.f;
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      // the lane's own particle in a padding slot: code 62 is offset 0
      const Offsets o = decode_code(ok[k] ? e[k] >> kCodeShift : 62u);
      float d0, d1, d2;
      rel_diff<DIM>(P, h, q[k], o, d0, d1, d2);
      const float r = __builtin_amdgcn_sqrtf(mixed_s2(d0, d1, d2));
      float w, gw;
      kernel_w_gradw_f32(P.kernel_type, r * P.inv_hf, P.coeff, P.coef_gradf, w, gw);
      if (ok[k]) acc.add(P.density_type == 1 ? mj[k] * w : w);
    }
  }
};

// Verlet lists: fixed-point positions, FP32 terms (without the kernel's factor
// coef) summed in FP64.  A candidate's in / out decision comes from its FP32
// distance, and in a band around the cut-off from the reference's FP64
// formula.
template <int DIM>
struct DensityMixed {
  const DevParams& P;
  const DeviceState& S;
  const Home& h;
  double acc;
  int nin = 0, rechecks = 0;
  static constexpr bool kImages = false;
  static constexpr bool kBatched = true;
  static constexpr int kBatch = 2;  // (larger ones cost the scan kernels registers)
  static constexpr int kTerms = 1;
  static constexpr int kWalk = 4;
  struct Rec {
    uint4 q;
    float mj;
  };
  __device__ __forceinline__ Rec gather(uint32_t ent) const {
    const uint32_t j = ent & kIndexMask;
    return {load_at(S.xq, j), P.density_type == 1 ? (float)S.m[j] : 1.f};
  }
  template <int NB>
  __device__ __forceinline__ void terms(const uint32_t (&e)[NB], const bool (&ok)[NB],
                                        Rec (&rec)[NB], double (&t)[NB][kTerms]) {
    const uint4 own = S.xq[h.ii];
    float s2[NB];
    bool use[NB];
    uint64_t band = 0;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      float d0, d1, d2;
      fixed_diff<DIM>(h, own, rec[k].q, d0, d1, d2);
      s2[k] = mixed_s2(d0, d1, d2);
      use[k] = ok[k] && s2[k] < P.cut2_lo_f32;
      band |= __ballot(s2[k] < P.cut2_hi_f32) & ~__ballot(s2[k] < P.cut2_lo_f32);
    }
    if (__builtin_expect(band != 0, 0)) {
#pragma unroll
      for (int k = 0; k < NB; ++k)
        if (ok[k])
          use[k] = mixed_inside<DIM>(P, S, h, (int)(e[k] & kIndexMask), s2[k], rechecks);
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      nin += use[k] ? 1 : 0;
      float w = kernel_w_f32(P.kernel_type, sqrt_refined(s2[k]) * P.inv_hf);
      if (P.density_type == 1) w = rec[k].mj * w;
      t[k][0] = (double)(use[k] ? w : 0.f);
    }
  }
  template <int NB>
  __device__ __forceinline__ void body_batch(const uint32_t (&e)[NB], const bool (&ok)[NB]) {
    double t[NB][kTerms];
    Rec rec[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) rec[k] = gather(e[k]);
    terms(e, ok, rec, t);
#pragma unroll
    for (int k = 0; k < NB; ++k) acc = acc + t[k][0];
  }
};

// Records of the force pass, written once the density is known.
//   FP64, Verlet lists: four planes of n 16-byte entries, (x, y), (z, p/n^2),
//   (vx, vy) and (vz, 1/n^2).  Neighbours in a list are near each other in
//   memory, so the lanes of a 16-byte gather share lines: gathers alone at the
//   128^3 box's lists take 151 CU cycles per wave-entry this way and 221 from
//   64-byte records (four lanes per particle).  The (x, y) plane follows the
//   positions (boundary, sort, track) and is not written here.
//   FP64, lists rebuilt every step: the same 64 bytes per particle together.  A
//   lane of that walk takes a whole list, and a record costs it four lines from
//   planes, one this way: forces of the 128^3 box 2.20 and 1.70 ms, 64^3 264 and
//   220 us, Oldroyd-B 64^3 434 and 354.
//   FP32 Newtonian: (cell-relative x, y, z, p/n^2 for Hu-Adams or p for the
//   angular form) and (vx, vy, vz, 1/n^2); the pair body gathers these two
//   and the particle id.
//   (Both FP32 forms: lists rebuilt every step.  Verlet lists: (v, 1/n^2),
//   p/n^2 or p apart, and for Oldroyd-B (Pxx, Pyy, Pzz, Pxy) and (Pxz, Pyz),
//   all but p with P.rec_scale; the position and pid are in xq.)
//   FP32 Oldroyd-B: (v, pid), (1/n^2, Pxx, Pyy, Pzz) and (Pxy, Pxz, Pyz, 0)
//   with P = Pi / n^2, Pi = (p + G) I - G c (particles_compute_pressure_
//   tensor.F90:114-133; c is symmetric); the position comes from xa.
template <int DIM>
__device__ __forceinline__ void write_force_records(const DevParams& P, const DeviceState& S, int i,
                                                    double an, double bn, double press) {
  const int64_t n = P.n;
  if (P.mixed) {
    const float v0 = (float)S.v[i], v1 = (float)S.v[n + i], v2 = DIM == 3 ? (float)S.v[2 * n + i] : 0.f;
    if (P.verlet) {
      S.vr[i] = make_float4(v0, v1, v2, (float)(bn * P.rec_scale));
      S.an32[i] = (float)(P.force_type == 4 ? press : an * P.rec_scale);
      if (!P.newtonian) {
        const double b = bn * P.rec_scale;
        auto pi = [&](int a, int c) {
          return (float)(((a == c ? press + P.G : 0.0) - P.G * S.ct[(int64_t)(a + DIM * c) * n + i]) * b);
        };
        S.qr[i] = make_float4(pi(0, 0), pi(1, 1), DIM == 3 ? pi(DIM - 1, DIM - 1) : 0.f, pi(0, 1));
        reinterpret_cast<float2*>(S.qr2)[i] =
            DIM == 3 ? make_float2(pi(0, DIM - 1), pi(1, DIM - 1)) : make_float2(0.f, 0.f);
      }
    } else if (P.newtonian) {
      const float4 xa = S.xa[i];
      S.qr[i] = make_float4(xa.x, xa.y, xa.z, (float)(P.force_type == 4 ? press : an));
      S.vr[i] = make_float4(v0, v1, v2, (float)bn);
    } else {
      S.vr[i] = make_float4(v0, v1, v2, __uint_as_float((uint32_t)S.pid[i]));
      auto pi = [&](int a, int b) {
        const double c = S.ct[(int64_t)(a + DIM * b) * n + i];
        return ((a == b ? press + P.G : 0.0) - P.G * c) * bn;
      };
      if (DIM == 3) {
        S.qr[i] = make_float4((float)bn, (float)pi(0, 0), (float)pi(1, 1), (float)pi(2, 2));
        S.qr2[i] = make_float4((float)pi(0, 1), (float)pi(0, 2), (float)pi(1, 2), 0.f);
      } else {
        S.qr[i] = make_float4((float)bn, (float)pi(0, 0), (float)pi(1, 1), 0.f);
        S.qr2[i] = make_float4((float)pi(0, 1), 0.f, 0.f, 0.f);
      }
    }
  } else {
    // entry q of the record is at pl[q * step]
    double2* pl = reinterpret_cast<double2*>(S.rec64) + (P.verlet ? i : 4 * (int64_t)i);
    const int64_t step = P.verlet ? n : 1;
    if (!P.verlet) pl[0] = make_double2(S.x[i], S.x[n + i]);
    pl[step] = make_double2(DIM == 3 ? S.x[2 * n + i] : 0.0, an);
    pl[2 * step] = make_double2(S.v[i], S.v[n + i]);
    pl[3 * step] = make_double2(DIM == 3 ? S.v[2 * n + i] : 0.0, bn);
    if (!P.newtonian) {
      // Oldroyd-B: Pi / n^2 as (xx, yy, zz, xy, xz, yz), Pi = (p + G) I - G c
      // (particles_compute_pressure_tensor.F90:114-133; c is symmetric)
      auto pib = [&](int a, int b) {
        const double c = S.ct[(int64_t)(a + DIM * b) * n + i];
        return ((a == b ? press + P.G : 0.0) - P.G * c) * bn;
      };
      double2* q = reinterpret_cast<double2*>(S.pt64) + (P.verlet ? i : 3 * (int64_t)i);
      if (DIM == 3) {
        q[0] = make_double2(pib(0, 0), pib(1, 1));
        q[step] = make_double2(pib(2, 2), pib(0, 1));
        q[2 * step] = make_double2(pib(0, 2), pib(1, 2));
      } else {
        q[0] = make_double2(pib(0, 0), pib(1, 1));
        q[step] = make_double2(0.0, pib(0, 1));
        q[2 * step] = make_double2(0.0, 0.0);
      }
    }
  }
}

// A chunk one of whose particles has more in-cutoff neighbours than the
// stored lists hold: its wave scans the stencil again in the force pass.
__device__ __forceinline__ bool list_overflow(const DevParams& P, const DeviceState& S,
                                              const Chunk& ch) {
  const int i = ch.p0 + (int)threadIdx.x;
  const int cnt = i < ch.p1 ? S.nbr_count[i] : 0;
  return __ballot(cnt > P.list_cap) != 0ull;
}

// Walk the in-cut-off pairs stored in a chunk's lists by the step's density
// pass (lists rebuilt every step; waves without list overflow).
template <int DIM, class Pol>
__device__ __forceinline__ void for_each_listed(const DevParams& P, const DeviceState& S,
                                                const Chunk& ch, const Home& h, Pol& pol,
                                                uint32_t* __restrict__ buf) {
  const int cnt = h.active ? S.nbr_count[h.i] : 0;
  const uint32_t* __restrict__ blk = list_block(P, S.nlist, ch);
  const int lane = threadIdx.x;
  for (int q = 0; __ballot(q < cnt) != 0ull; q += 8) {
    if (q < cnt) {
      // eight entries per pair of 16-byte loads; entries past cnt are
      // padding inside the row and are not evaluated.  The group goes to
      // LDS (entry u of a lane at buf[u * 64 + lane], conflict-free), and
      // the loop reads one entry per pair, the next one ahead of the body.
      const uint4* src = reinterpret_cast<const uint4*>(blk + group_offset(ch, q, lane));
      const uint4 lo = src[0], hi = src[1];
      buf[0 * kWave + lane] = lo.x;
      buf[1 * kWave + lane] = lo.y;
      buf[2 * kWave + lane] = lo.z;
      buf[3 * kWave + lane] = lo.w;
      buf[4 * kWave + lane] = hi.x;
      buf[5 * kWave + lane] = hi.y;
      buf[6 * kWave + lane] = hi.z;
      buf[7 * kWave + lane] = hi.w;
      const int m = min(8, cnt - q);
      uint32_t ent = buf[lane];
#pragma unroll 1
      for (int u = 0; u < m; ++u) {
        const uint32_t cur = ent;
        ent = buf[((u + 1) & 7) * kWave + lane];
        pol.body(cur);
      }
    }
  }
}

// ---------------------------------------------------------------------
// the walk of Verlet lists: four or sixteen lanes per particle
// ---------------------------------------------------------------------
// A wave takes 64 / LANES consecutive particles of a chunk (a "part"), a lane
// every LANES-th entry of one particle.  Against one particle per lane,
// neighbouring lanes gather neighbouring list entries (fewer lines per
// gather), a wave runs as long as the longest of 16 (4) lists instead of 64,
// and a small box has 4 (16) times the waves, each as much shorter.
//
// The terms are still added in list order: a group's lanes put their terms
// into LDS, and lane s of a particle adds component s (with four lanes also
// 4 + s, 8 + s) of its entries one after another.  So a particle's sum does not
// depend on where its in-cut-off pairs stand among the candidates, and equals
// the one-particle-per-lane sums of the candidate scans bit for bit.  With four
// lanes four FP64 adds per four components and 64 entries; the matrix cores'
// v_mfma_f64_4x4x4 (an fma chain over k, the same order) takes 4 CU cycles per
// component, and on the 128^3 box the force walk took 1.54 ms with it.  With
// sixteen lanes 16 adds per 64 entries, and a prologue for every 4 particles.
template <int LANES>
constexpr int kPart = kWave / LANES;  // particles of a wave
// a component's row of 64 lanes' terms: 66 doubles, so that the 16-byte reads
// of the four lanes' rows fall on different banks
constexpr int kTermRow = 66;
template <int TERMS>
constexpr int kTermRows = (TERMS + 3) / 4 * 4 * kTermRow;
// (sixteen lanes: entries 0 .. 3 of the groups and entries 4 .. 7)
template <int TERMS, int LANES>
constexpr int kTermWords = kTermRows<TERMS> * (LANES == 16 ? 2 : 1);

// the sums of a wave's particles after the walk: component c of particle p
__device__ __forceinline__ double& part_sum(double* lds, int p, int c) {
  return lds[c * kTermRow + p];
}

// start: what the sum of component 0 starts from (a particle's first lane).
// Leaves the sums in lds (part_sum).
template <int DIM, int LANES, class Pol>
__device__ __forceinline__ void walk_part(const DevParams& P, const DeviceState& S,
                                          const Chunk& ch, int part, const Home& h, Pol& pol,
                                          double start, double* __restrict__ lds) {
  static_assert(LANES == 4 || LANES == 16, "");
  constexpr int NB = LANES == 4 ? Pol::kWalk : 2;  // entries per lane and batch (even)
  constexpr int T = Pol::kTerms, M = (T + LANES - 1) / LANES;
  constexpr int kGroups = LANES / 4;  // list groups of 8 that two of a lane's entries span
  const int lane = threadIdx.x;
  const int s = lane & (LANES - 1), p = lane / LANES;
  const int s4 = s & 3, gl = s >> 2;
  const int cnt = h.active ? S.nbr_count[h.i] : 0;
  const uint32_t* __restrict__ src =
      list_block(P, S.nlist, ch) + (kPart<LANES> * part + p) * 8 + 2 * s4;
  double* __restrict__ put = lds + lane;
  // (lanes past the components repeat the last one's sum, unused)
  const double2* __restrict__ get = reinterpret_cast<const double2*>(
      lds + (LANES == 4 ? s : min(s, T - 1)) * kTermRow + LANES * p);
  double sum[M];
#pragma unroll
  for (int m = 0; m < M; ++m) sum[m] = 0.0;
  if (s == 0) sum[0] = start;
  // the next batch's entries are loaded behind the current batch's gathers,
  // without a branch (a group past the list's capacity reads its last one)
  const int last = (P.list_cap >> 3) - 1, stride = (ch.p1 - ch.p0) * 8;
  uint2 nx[NB / 2];
  auto fetch = [&](int q) {
#pragma unroll
    for (int g = 0; g < NB / 2; ++g)
      nx[g] = *reinterpret_cast<const uint2*>(
          src + min((q >> 3) + g * kGroups + gl, last) * stride);
  };
  fetch(0);
  for (int q = 0; __ballot(q < cnt) != 0ull; q += LANES * NB) {
    uint32_t e[NB];
    bool ok[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      ok[k] = q + 8 * (k / 2 * kGroups + gl) + 4 * (k & 1) + s4 < cnt;
      e[k] = ok[k] ? ((k & 1) ? nx[k / 2].y : nx[k / 2].x) : (uint32_t)h.ii;
    }
    typename Pol::Rec r[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) r[k] = pol.gather(e[k]);
    fetch(q + LANES * NB);
    // (the density bodies are short: the scheduler would sink some of these
    // loads to their first use, one wait each -- the FP64 walk of the 128^3
    // box takes 0.78 instead of 0.58 ms then)
    if constexpr (T == 1) __builtin_amdgcn_sched_barrier(0);
    double t[NB][T];
    pol.terms(e, ok, r, t);
    // (one wave per workgroup: its LDS operations complete in order)
    if constexpr (LANES == 4) {
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int c = 0; c < T; ++c) put[c * kTermRow] = t[k][c];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const double2 a = get[2 * m * kTermRow], b = get[2 * m * kTermRow + 1];
          sum[m] = sum[m] + a.x;
          sum[m] = sum[m] + a.y;
          sum[m] = sum[m] + b.x;
          sum[m] = sum[m] + b.y;
        }
      }
    } else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int c = 0; c < T; ++c) put[k * kTermRows<T> + c * kTermRow] = t[k][c];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int g = 0; g < kGroups; ++g)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const double2 a = get[k * kTermRows<T> / 2 + 2 * g];
          const double2 b = get[k * kTermRows<T> / 2 + 2 * g + 1];
          sum[0] = sum[0] + a.x;
          sum[0] = sum[0] + a.y;
          sum[0] = sum[0] + b.x;
          sum[0] = sum[0] + b.y;
        }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int m = 0; m < M; ++m)
    if (LANES == 4 || s < T) part_sum(lds, p, LANES * m + s) = sum[m];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// The home particle of a lane in the walk of a part.
template <int DIM, int LANES>
__device__ __forceinline__ Home load_part_home(const DevParams& P, const DeviceState& S,
                                               const Chunk& ch, int part) {
  Home h;
  h.i = ch.p0 + kPart<LANES> * part + (int)threadIdx.x / LANES;
  h.active = h.i < ch.p1;
  h.ii = h.active ? h.i : ch.p0;
  const int64_t n = P.n;
  h.G = ch.G;
  h.cx = (S.key_sorted[h.ii] - ch.G.cell_base) % ch.G.nm0;
  const int lr = ch.row - ch.G.row_base;
  h.cy = lr % ch.G.nm1;
  h.cz = lr / ch.G.nm1;
  h.a = S.xa[h.ii];
  h.x0 = S.x[h.ii];
  h.x1 = S.x[n + h.ii];
  h.x2 = DIM == 3 ? S.x[2 * n + h.ii] : 0.0;
  if (P.le_g >= 0) {
    h.le.t = S.time_dev[1];
    h.le.sp0 = f_modulo((P.le_vhi - P.le_vlo) * h.le.t, ch.G.L0);
    h.le.sp1 = f_modulo((P.le_vlo - P.le_vhi) * h.le.t, ch.G.L0);
  }
  return h;
}

// Chunk slot of a workgroup and which of the chunk's G workgroups it is: they
// are 8 apart, so they share an XCD.
template <int G>
__device__ __forceinline__ int part_slot(int b, int& which) {
  which = (b / 8) % G;
  return b / (8 * G) * 8 + b % 8;
}

// Whether a chunk's row of cells lies within `cells` cells of a face of
// dimension le_g (2: its stencil rows reach across the face).
__device__ __forceinline__ bool chunk_meets_le_face(int le_g, const Chunk& ch, int cells) {
  const int lr = ch.row - ch.G.row_base;
  const int c = le_g == 1 ? lr % ch.G.nm1 : lr / ch.G.nm1;
  const int nm = le_g == 1 ? ch.G.nm1 : ch.G.nm2;
  return c < cells || c >= nm - cells;
}

// LE = false compiles the Lees-Edwards paths out: le_g is then the
// constant -1 in every inlined helper.  A box with sheared faces runs two
// launches over the same grid, LE = true for the chunks next to a face and
// LE = false for the rest, whose rows never cross a face (the sheared
// frame's state would cost the whole pass registers and occupancy).
//
// Modes.  kStore: the in-cut-off pairs found by the candidate scan are
// summed and stored (lists rebuilt every step).  Verlet lists decide the
// cut-off per candidate on the current positions: k_density_walk walks the
// lists of the chunks that hold them all, and kScan, before it, stores the
// candidates within rc + skin of every chunk on steps whose gate asks for it,
// and scans the stencil for the sums of the chunks whose lists overflowed.  The
// walk and the scans visit the candidates in the same order, so they give the
// same sums.
enum DensityMode { kStore = 0, kScan = 1 };

// The pressure of particle i and its factors of the pair forces: p/n^2 and 1/n^2
// (Newtonian Morris and Espanol, whose viscous terms divide by n_i n_j: 1/n).
__device__ __forceinline__ void store_pressure(const DevParams& P, const DeviceState& S, int i,
                                               double rho, double press, double& an, double& bn) {
  an = press / (rho * rho);
  bn = (P.newtonian && P.force_type <= 2) ? 1.0 / rho : 1.0 / (rho * rho);
  S.p[i] = press;
  S.an[i] = an;
  S.bn[i] = bn;
}

// Density epilogue of particle i with number (or mass) density sum rho.
template <int DIM>
__device__ __forceinline__ void finish_density(const DevParams& P, const DeviceState& S, int i,
                                               double mi, double rho, int nin, int rechecks) {
  // colloid boundary particles of constant density take the initial
  // density rho (number density rho / m) instead of the sum
  // (particles_compute_density.F90:442-473, 526-556)
  if (P.ncoll && P.coll_rho_type == 0 && S.sid[i] != 0)
    rho = P.density_type == 1 ? P.rho0 : P.rho0 / mi;
  const double press = eos_pressure(P, P.density_type == 2 ? rho * mi : rho);
  S.rho[i] = rho;
  double an, bn;
  store_pressure(P, S, i, rho, press, an, bn);
  S.nbr_in[i] = nin;
  S.recheck[i] = rechecks;
  write_force_records<DIM>(P, S, i, an, bn, press);
}

// The self term that starts a particle's density sum
// (particles_compute_density.F90:369-558).
template <bool MIXED>
__device__ __forceinline__ double self_density(const DevParams& P, double mi) {
  // (the sums leave the kernel's factor to density_of)
  const double w = MIXED ? P.w0 / P.coef : P.w0q;
  return P.density_type == 1 ? w * mi : w;
}
template <bool MIXED>
__device__ __forceinline__ double density_of(const DevParams& P, double sum) {
  return (MIXED ? P.coef : P.cw) * sum;
}

// The density sums of a chunk by a scan of the stencil.
template <int DIM, bool MIXED, int TILE, int BUF, int MODE>
__device__ __forceinline__ void scan_density(const DevParams& P, const DeviceState& S,
                                             const Chunk& ch, const Home& h,
                                             float4* __restrict__ tile,
                                             uint32_t* __restrict__ buf, bool store) {
  constexpr bool kDecide = MODE != kStore;
  const double mi = S.m[h.ii];
  uint32_t* list = MODE == kStore ? S.nlist : nullptr;
  using Pol = std::conditional_t<
      MIXED, std::conditional_t<kDecide, DensityMixed<DIM>, DensityMixedStep<DIM>>,
      DensityF64<DIM, kDecide>>;
  Pol pol{P, S, h, {}};
  if constexpr (MIXED && !kDecide)
    pol.acc.add((float)(P.density_type == 1 ? P.w0 * mi : P.w0));
  else
    pol.acc = self_density<MIXED>(P, mi);
  int rechecks = 0;
  const int cnt =
      staged_scan<DIM, Pol, TILE, BUF, kDecide>(P, S, ch, h, pol, tile, buf, rechecks, list);
  double rho;
  if constexpr (MIXED && !kDecide)
    rho = pol.acc.value();
  else
    rho = density_of<MIXED>(P, pol.acc);
  if (!h.active || !store) return;
  const int i = h.i;
  if (MODE == kStore) S.nbr_count[i] = cnt;
  finish_density<DIM>(P, S, i, mi, rho, kDecide ? pol.nin : cnt, rechecks + pol.rechecks);
}

// One chunk slot of a density pass that scans the stencil.
template <int DIM, bool MIXED, int TILE, int BUF, bool LE, int MODE>
__device__ __forceinline__ void density_chunk(const DevParams& P, const DeviceState& S, int slot,
                                              int le_box, bool build,
                                              float4* __restrict__ tile,
                                              uint32_t* __restrict__ buf) {
  Chunk ch;
  if (!load_chunk(P, S, ch, slot)) return;
  if (le_box >= 0 && chunk_meets_le_face(le_box, ch, 2) != LE) return;
  if (MODE == kScan && !build && !list_overflow(P, S, ch)) return;
  const Home h = load_home<DIM>(P, S, ch);
  if (MODE == kScan && build) {
    const int cnt = list_scan<DIM, !MIXED, TILE, BUF>(P, S, ch, h, ch.p1 - ch.p0, threadIdx.x, tile,
                                                      buf, list_block(P, S.nlist, ch));
    if (h.active) S.nbr_count[h.i] = cnt;
    // the shear time of the build (the copies across sheared faces drift
    // from their build positions as it advances)
    if (h.active && h.i == 0) S.time_dev[3] = S.time_dev[1];
    if (__ballot(h.active && cnt > P.list_cap) == 0ull) return;
    if (threadIdx.x == 0) S.gate[2] = 1;  // every writer stores 1
  }
  scan_density<DIM, MIXED, TILE, BUF, MODE>(P, S, ch, h, tile, buf, true);
}

// The build of small boxes: a workgroup of four waves per chunk, 16 particles
// each, so that a wave's chain of rows is shorter and there are four times as
// many.  The chunk's waves sum overflowed lists alike, each in its own LDS, and
// the first one stores.
template <int DIM, bool MIXED>
__global__ __launch_bounds__(4 * kWave, 4) void k_density_split(DevParams P, DeviceState S) {
  const bool build = S.gate[0] != 0;
  if (!build && S.gate[2] == 0) return;
  P.le_g = -1;
  __shared__ float4 tiles[4][kTile + kTilePad<4>];
  __shared__ uint32_t bufs[4][kBuf * kWave];
  __shared__ int over;
  const int wave = threadIdx.y;
  float4* __restrict__ tile = tiles[wave];
  uint32_t* __restrict__ buf = bufs[wave];
  const int slots = chunk_slots(P);
  for (int slot = blockIdx.x; slot < slots; slot += gridDim.x) {
    Chunk ch;
    if (!load_chunk(P, S, ch, slot)) continue;
    if (build) {
      if (wave == 0 && threadIdx.x == 0) over = 0;
      __syncthreads();
      Chunk own = ch;
      own.p0 = ch.p0 + kPart<4> * wave;
      own.p1 = min(own.p0 + kPart<4>, ch.p1);
      if (own.p0 < own.p1) {
        own.xmin = (S.key_sorted[own.p0] - ch.G.cell_base) % ch.G.nm0;
        own.xmax = (S.key_sorted[own.p1 - 1] - ch.G.cell_base) % ch.G.nm0;
        const Home h = load_part_home<DIM, 4>(P, S, ch, wave);
        const int cnt = list_scan<DIM, !MIXED, kTile, kBuf, 4>(
            P, S, own, h, ch.p1 - ch.p0, kPart<4> * wave + (int)threadIdx.x / 4, tile, buf,
            list_block(P, S.nlist, ch));
        if (h.active && (threadIdx.x & 3) == 0) S.nbr_count[h.i] = cnt;
        if (h.active && h.i == 0) S.time_dev[3] = S.time_dev[1];
        if (h.active && cnt > P.list_cap) over = 1;  // every writer stores 1
      }
      __syncthreads();
      const bool scan = over != 0;
      __syncthreads();
      if (!scan) continue;
      if (threadIdx.x == 0) S.gate[2] = 1;
    } else if (!list_overflow(P, S, ch)) {
      continue;
    }
    scan_density<DIM, MIXED, kTile, kBuf, kScan>(P, S, ch, load_home<DIM>(P, S, ch), tile, buf,
                                                 wave == 0);
    __syncthreads();
  }
}

// The walk of the step's Verlet lists: NQ parts of a chunk per workgroup.
// Quarters of a chunk one after the other let the epilogue (equation of state,
// force records) run once on 64 lanes (128^3 box: FP64 0.58 ms, 0.65 with one
// quarter per workgroup; mixed 0.46 and 0.49); a small box takes one part per
// workgroup to fill the GPU.  QUINTIC: the quintic spline and the number density
// as constants, so the batch's terms carry no branches.
template <int DIM, bool MIXED, bool LE, bool QUINTIC, int NQ, int LANES>
__global__ __launch_bounds__(kWave) void k_density_walk(DevParams P, DeviceState S) {
  // the lists are current, and no force walk has left the scan anything yet
  if (blockIdx.x == 0 && threadIdx.x == 0) S.gate[0] = S.gate[4] = 0;
  __shared__ __align__(16) double lds[kTermWords<1, LANES>];
  constexpr int kOwn = kPart<LANES>;
  const int le_box = P.le_g;
  if (!LE) P.le_g = -1;
  if (QUINTIC) {
    P.kernel_type = 1;
    P.density_type = 2;
  }
  int q0;
  Chunk ch;
  if (!load_chunk(P, S, ch, part_slot<LANES / NQ>(blockIdx.x, q0))) return;
  q0 *= NQ;
  if (ch.p0 + kOwn * q0 >= ch.p1) return;
  if (le_box >= 0 && chunk_meets_le_face(le_box, ch, 2) != LE) return;
  if (S.gate[2] != 0 && list_overflow(P, S, ch)) return;
  const int lane = threadIdx.x;
  double rho = 0.0;
  int nin = 0, rechecks = 0;
#pragma unroll 1
  for (int q = 0; q < NQ && ch.p0 + kOwn * (q0 + q) < ch.p1; ++q) {
    const Home h = load_part_home<DIM, LANES>(P, S, ch, q0 + q);
    using Pol = std::conditional_t<MIXED, DensityMixed<DIM>, DensityF64<DIM, true>>;
    Pol pol{P, S, h, {}};
    walk_part<DIM, LANES>(P, S, ch, q0 + q, h, pol,
                          self_density<MIXED>(P, QUINTIC ? 1.0 : S.m[h.ii]), lds);
    int in = pol.nin, re = pol.rechecks;
#pragma unroll
    for (int off = 1; off < LANES; off *= 2) {
      in += __shfl_xor(in, off);
      re += __shfl_xor(re, off);
    }
    const double r = part_sum(lds, lane & (kOwn - 1), 0);
    in = __shfl(in, LANES * (lane & (kOwn - 1)));
    re = __shfl(re, LANES * (lane & (kOwn - 1)));
    if (lane / kOwn == q) {
      rho = r;
      nin = in;
      rechecks = re;
    }
  }
  const int i = ch.p0 + kOwn * q0 + lane;
  if (lane >= kOwn * NQ || i >= ch.p1) return;
  finish_density<DIM>(P, S, i, S.m[i], density_of<MIXED>(P, rho), nin, rechecks);
}

// kScan has work only when the lists are built or one overflowed then: its
// workgroups take every gridDim.x-th chunk slot, so that on the other steps
// the launch is cheap.
template <int DIM, bool MIXED, int TILE, int BUF, bool LE, int MODE>
__global__ __launch_bounds__(kWave, MODE == kScan ? 4 : 1) void k_density(DevParams P, DeviceState S) {
  const bool build = MODE == kScan && S.gate[0] != 0;
  if (MODE == kScan && !build && S.gate[2] == 0) return;
  const int le_box = P.le_g;
  if (!LE) P.le_g = -1;
  __shared__ float4 tile[TILE + 3];
  // whole groups of 8 rows: the final flush stores the last group of a
  // lane's entries as 8 rows, of which those past its count are padding
  __shared__ uint32_t buf[(BUF + 7) / 8 * 8 * kWave];
  if (MODE == kScan) {
    const int slots = chunk_slots(P);
    for (int slot = blockIdx.x; slot < slots; slot += gridDim.x) {
      density_chunk<DIM, MIXED, TILE, BUF, LE, MODE>(P, S, slot, le_box, build, tile, buf);
      __syncthreads();
    }
  } else {
    density_chunk<DIM, MIXED, TILE, BUF, LE, MODE>(P, S, blockIdx.x, le_box, false, tile, buf);
  }
}

__global__ void k_eos(DevParams P, DeviceState S) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  const double r = S.rho[i];
  double an, bn;
  store_pressure(P, S, i, r, eos_pressure(P, P.density_type == 2 ? r * S.m[i] : r), an, bn);
}

// Force-pass records after the velocities or the pressure changed between
// the density and the force pass (separate kick / EOS calls).
__global__ void k_refresh_records(DevParams P, DeviceState S) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  if (P.dim == 3)
    write_force_records<3>(P, S, i, S.an[i], S.bn[i], S.p[i]);
  else
    write_force_records<2>(P, S, i, S.an[i], S.bn[i], S.p[i]);
}

// ---------------------------------------------------------------------
// K4: pair forces
// ---------------------------------------------------------------------

// Random force direction seen by particle i for neighbour j: a Gaussian
// vector with the covariance of the reference's symmetric traceless
// dW . e_ij (I/2 + e e^T/6 in 3D, I/2 in 2D), oriented by the lower pid.
// g3 (Espanol's trace draw): the block's fourth normal, shared by the pair.
template <int DIM, typename T>
__device__ __forceinline__ void noise_vector(const DevParams& P, int64_t step, uint32_t pidi,
                                             uint32_t pidj, T e0, T e1, T e2, T& w0, T& w1,
                                             T& w2, T* g3 = nullptr) {
  uint32_t lo = pidi < pidj ? pidi : pidj, hi = pidi < pidj ? pidj : pidi;
  float g[4];
  pair_normals(P.seed, lo, hi, step, g);
  if (g3) *g3 = (T)g[3];
  const T sgn = pidi < pidj ? T(1) : T(-1);
  const T ca = T(0.70710678118654752440);
  if (DIM == 3) {
    const T cb = T(0.81649658092772603273) - T(0.70710678118654752440);
    T c0 = sgn * e0, c1 = sgn * e1, c2 = sgn * e2;
    T ge = (T)g[0] * c0 + (T)g[1] * c1 + (T)g[2] * c2;
    w0 = sgn * (ca * (T)g[0] + cb * ge * c0);
    w1 = sgn * (ca * (T)g[1] + cb * ge * c1);
    w2 = sgn * (ca * (T)g[2] + cb * ge * c2);
  } else {
    w0 = sgn * (ca * (T)g[0]);
    w1 = sgn * (ca * (T)g[1]);
    w2 = T(0);
  }
}

// One FP64 force record, gathered from its four planes (Verlet lists) or from its
// 64 bytes.
struct RecF64 {
  double2 a, b, c, d;  // (x, y), (z, p/n^2), (vx, vy), (vz, 1/n^2)
  uint32_t pid;        // with thermal noise, from the planes
  double2 q0, q1, q2;  // Oldroyd-B: Pi / n^2 as (xx, yy), (zz, xy), (xz, yz)
};
template <bool TENSOR, bool PLANES>
__device__ __forceinline__ RecF64 load_rec(const DevParams& P, const DeviceState& S, uint32_t j) {
  const double2* __restrict__ pl = reinterpret_cast<const double2*>(S.rec64);
  const int64_t n = P.n;
  RecF64 r;
  if (!PLANES) {
    const double2* __restrict__ one = pl + 4 * (int64_t)j;
    r.a = one[0];
    r.b = one[1];
    r.d = one[3];
    r.c = one[2];
    // (before anything else: 128^3 1.85 ms without)
    __builtin_amdgcn_sched_barrier(0);
    r.pid = 0u;
    if (TENSOR) {
      const double2* __restrict__ pt = reinterpret_cast<const double2*>(S.pt64) + 3 * (int64_t)j;
      r.q0 = pt[0];
      r.q1 = pt[1];
      r.q2 = pt[2];
    }
    return r;
  }
  r.a = load_at(pl, j);
  r.b = load_at(pl + n, j);
  r.c = load_at(pl + 2 * n, j);
  r.d = load_at(pl + 3 * n, j);
  r.pid = P.noise ? (uint32_t)load_at(S.pid, j) : 0u;
  if (TENSOR) {
    const double2* __restrict__ pt = reinterpret_cast<const double2*>(S.pt64);
    r.q0 = load_at(pt, j);
    r.q1 = load_at(pt + n, j);
    r.q2 = load_at(pt + 2 * n, j);
  }
  return r;
}

// The pair bodies of Verlet lists without colloids (kStraight) take no in / out
// decision: a candidate outside the cut-off adds its kernel gradient, 0, times
// the rest.  That is 0 only while the rest is finite.  A wave whose sums do not
// all come out finite (a velocity, pressure or tensor of a neighbour, a
// candidate or the particle itself is not) sums again, or leaves its chunk to the
// scan of overflowed lists, with bodies (LEAVE) that leave out the candidates
// outside the cut-off, as the reference does.
__device__ __forceinline__ bool not_finite(double a) { return !(fabs(a) < __builtin_inf()); }
// the terms of the lanes in out become 0
template <int NB, int T, class F>
__device__ __forceinline__ void leave_out(const uint64_t (&out)[NB], F (&t)[NB][T]) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int k = 0; k < NB; ++k)
#pragma unroll
    for (int c = 0; c < T; ++c) t[k][c] = ((out[k] >> lane) & 1) != 0 ? F(0) : t[k][c];
}

// force types: 3 Hu-Adams, 4 Hu-Adams angular, 5 Oldroyd-B (non-Newtonian
// Hu-Adams).  The bodies sum m_i times the acceleration (and the Oldroyd-B
// velocity gradient); finish_force divides by m_i once.  DECIDE (Verlet
// lists): the entries are candidates within rc + skin; those outside the
// cut-off add 0.
template <int DIM, int FT, bool COLL = false, bool DECIDE = false, bool LEAVE = false>
struct ForceF64 {
  const DevParams& P;
  const DeviceState& S;
  const Home& h;
  double vi0, vi1, vi2, ai, bi, pi, inv_ni;
  uint32_t pidi;
  int64_t step;            // noise step (the context's marching step)
  // the acceleration's components, then the velocity gradient's
  static constexpr int kTerms = DIM + (FT >= 5 ? DIM * DIM : 0);
  double sum[kTerms];
  // kUnit: the terms leave out the factor cg of the kernel gradient, and the
  // velocity gradient's leave out 1 / n_i (not around colloids): finish_pairs
  static constexpr bool kUnit = FT == 3 || FT == 5;
  // Oldroyd-B: own Pi / n_i^2 (Pi for the angular form)
  double pti[9];
  // colloids: own species id; a boundary particle's position relative to
  // the nearest image of its colloid's centre and that image's velocity;
  // time of the pass's shear length
  int sidi = 0;
  double rxc_i[3] = {0.0, 0.0, 0.0}, vcoll_i[3] = {0.0, 0.0, 0.0};
  double le_t = 0.0;
  static constexpr bool kImages = true;
  static constexpr bool kBatched = DECIDE;
  static constexpr int kBatch = 2;
  static constexpr int kWalk = 2;
  // fluid pairs of Verlet lists need no in / out decision of their own:
  // outside the cut-off the kernel gradient is 0
  static constexpr bool kStraight = DECIDE && !COLL;
  __device__ __forceinline__ void body(uint32_t ent) {
    const uint32_t j = ent & kIndexMask;
    if (COLL) {
      // two boundary particles do not interact (pp_interaction.inc: same
      // colloid CYCLE, colloid-colloid pair forces off)
      if (sidi != 0 && (ent & kBoundaryBit) != 0u) return;
    }
    const RecF64 r = load_rec<(FT >= 5), DECIDE>(P, S, j);
    const Images o = decode_images(ent);
    double d0, d1, d2;
    const double r2 = pair_d2<DIM>(P, h, o, r.a.x, r.a.y, r.b.x, d0, d1, d2);
    double t[kTerms];
    eval(ent, r, d0, d1, d2, r2, le_dv(P, o), t);
#pragma unroll
    for (int c = 0; c < kTerms; ++c) sum[c] = sum[c] + t[c];
  }
  template <int NB>
  __device__ __forceinline__ void body_batch(const uint32_t (&e)[NB], const bool (&ok)[NB]) {
    double t[NB][kTerms];
    Rec r[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) r[k] = gather(e[k]);
    terms(e, ok, r, t);
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
      for (int c = 0; c < kTerms; ++c) sum[c] = sum[c] + t[k][c];
  }
  using Rec = RecF64;
  __device__ __forceinline__ Rec gather(uint32_t ent) const {
    return load_rec<(FT >= 5), true>(P, S, ent & kIndexMask);
  }
  // The terms of NB candidates, whose records are gathered already.
  template <int NB>
  __device__ __forceinline__ void terms(const uint32_t (&e)[NB], const bool (&ok)[NB],
                                        Rec (&r)[NB], double (&t)[NB][kTerms]) const {
    if constexpr (kStraight) {
      auto square = [](double a, double b, double c) {
        return DIM == 3 ? fma(c, c, fma(b, b, a * a)) : fma(b, b, a * a);
      };
      // the plain differences, a branch of the wave for the batches with a
      // pair across a face and one for those with an empty slot: the pairs
      // are then evaluated without branches
      double d[NB][3], r2[NB];
      uint64_t far = 0, empty = 0;
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        d[k][0] = h.x0 - r[k].a.x;
        d[k][1] = h.x1 - r[k].a.y;
        d[k][2] = DIM == 3 ? h.x2 - r[k].b.x : 0.0;
        r2[k] = square(d[k][0], d[k][1], d[k][2]);
        far |= __ballot(!(r2[k] <= h.G.half2));
        empty |= __ballot(!ok[k]);
      }
      if (__builtin_expect(far != 0, 0)) {
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          double jump = 0.0;
          if (nearest_image<DIM>(P, h, d[k][0], d[k][1], d[k][2], jump)) {
            if (P.le_g >= 0) r[k].c.x = r[k].c.x + jump;
          } else {
            // (no velocity difference either, should j's be NaN as well)
            r[k].c = make_double2(vi0, vi1);
            r[k].d.x = vi2;
          }
          r2[k] = square(d[k][0], d[k][1], d[k][2]);
        }
      }
      uint64_t out[NB] = {};
      if constexpr (LEAVE) {
#pragma unroll
        for (int k = 0; k < NB; ++k) out[k] = __ballot(!(ok[k] && r2[k] < P.cut2));
      }
      // an empty slot holds the lane's own particle, no separation and no
      // velocity difference: at a squared distance outside the cut-off it
      // adds 0
      if (__builtin_expect(empty != 0, 0)) {
#pragma unroll
        for (int k = 0; k < NB; ++k) r2[k] = ok[k] ? r2[k] : 4.0 * P.cut2;
      }
#pragma unroll
      for (int k = 0; k < NB; ++k)
        eval(e[k], r[k], d[k][0], d[k][1], d[k][2], r2[k], 0.0, t[k]);
      if constexpr (LEAVE) leave_out(out, t);
    } else {
#pragma unroll
      for (int k = 0; k < NB; ++k) {
#pragma unroll
        for (int c = 0; c < kTerms; ++c) t[k][c] = 0.0;
        // two boundary particles do not interact
        if (!ok[k] || (COLL && sidi != 0 && (e[k] & kBoundaryBit) != 0u)) continue;
        // the image and the sheared face crossed come from the positions
        double d0, d1, d2;
        int sg;
        const double r2 =
            exact_d2_verlet<DIM>(P, h, r[k].a.x, r[k].a.y, r[k].b.x, d0, d1, d2, sg);
        if (!(r2 < P.cut2)) continue;
        eval(e[k], r[k], d0, d1, d2, r2, sg == 0 ? P.le_u : (sg == 1 ? -P.le_u : 0.0), t[k]);
      }
    }
  }
  // The terms of one pair: j's record, the separation d and its square, the
  // x velocity of j's image minus j's own.
  __device__ __forceinline__ void eval(uint32_t ent, const RecF64& rj, double d0, double d1,
                                       double d2, double r2, double jump,
                                       double (&t)[kTerms]) const {
    const int j = (int)(ent & kIndexMask);
    // j's pid, where the noise needs it.  Lists rebuilt every step gather it there,
    // not with the record: a wave that asked for both at once, and so went on
    // sooner, had its lines taken from the L1 by others' (128^3 2.04 and 1.72 ms).
    auto pid_j = [&]() {
      if constexpr (DECIDE) return rj.pid;
      __builtin_amdgcn_sched_barrier(0);
      return (uint32_t)S.pid[j];
    };
    const bool jb = COLL && (ent & kBoundaryBit) != 0u;
    const double ir = rsqrt_nr(r2);
    const double r = r2 * ir;
    const double gw = kUnit ? kernel_g(P, r) : P.cg * kernel_g(P, r);
    // (without sheared faces the jump is the constant 0 and no add is made)
    double u0 = vi0 - (P.le_g >= 0 && !kStraight ? rj.c.x + jump : rj.c.x), u1 = vi1 - rj.c.y,
           u2 = DIM == 3 ? vi2 - rj.d.x : 0.0;
    const double an = rj.b.y, bj = rj.d.y;
    // pressure terms: p_i / n_i^2 + p_j / n_j^2 (type 3), (p_i + p_j) / 2 (type 4)
    double psum = 0.0, pij = 0.0;
    if (FT <= 3) psum = ai + an;
    if (FT == 4) pij = (pi + S.p[j]) * 0.5;
    // with a colloid boundary particle in an Oldroyd-B flow both sides take
    // the fluid particle's 1/n^2 and Pi/n^2
    // (pp_interaction_fc.inc:80-113, pp_interaction_cf.inc:80-110)
    double bsum = bi + bj;
    const bool cpair = COLL && (sidi != 0 || jb);
    if (cpair) {
      // a fluid particle and a colloid boundary particle: the boundary
      // particle's velocity changes, and its pressure (Newtonian) or its
      // number density and pressure tensor (Oldroyd-B)
      double pb;
      colloid_substitute(j, jb ? S.sid[j] : 0, rj, d0, d1, d2, jump, u0, u1, u2, pb);
      if (FT == 3) psum = sidi == 0 ? ai + pb * bj : pb * bi + an;
      // Morris and Espanol: bi, bj = 1/rho
      if (FT <= 2) psum = sidi == 0 ? ai + pb * (bj * bj) : pb * (bi * bi) + an;
      if (FT == 4) pij = pb;
      if (FT == 5) bsum = sidi == 0 ? bi + bi : bj + bj;
    }
    double a0, a1, a2;
    if (FT == 1) {
      // rhs_force_ff_Newtonian_Morris.F90:112-136: accelerations, each term
      // carrying the partner's mass (the caller skips the division by m_i);
      // bi, bj = 1/rho
      const double mj = S.m[j];
      const double fcm = mj * psum * gw * ir;
      const double fdm = mj * 2.0 * P.eta * gw * bi * bj * ir;
      a0 = fdm * u0 - fcm * d0;
      a1 = fdm * u1 - fcm * d1;
      a2 = fdm * u2 - fcm * d2;
    } else if (FT == 2) {
      // rhs_force_ff_Newtonian_Espanol.F90:152-251; bi, bj = 1/n
      const double gnn = gw * bi * bj * ir;
      const double ev = (DIM == 3 ? fma(d2, u2, fma(d1, u1, d0 * u0)) : fma(d1, u1, d0 * u0)) * ir;
      const double fd1 = (2.0 - 1.0 / DIM) * P.eta * gnn;
      const double fd2 = P.eta * (DIM + 2.0) / DIM * gnn * ev;
      // pressure and the dissipative term along e, both along d / r
      const double se = (psum * gw * -1.0 + fd2) * ir;
      a0 = fd1 * u0 + se * d0;
      a1 = fd1 * u1 + se * d1;
      a2 = fd1 * u2 + se * d2;
      if (P.noise) espanol_noise(pid_j(), d0, d1, d2, ir, gnn, a0, a1, a2);
    } else if (FT == 4) {
      // rhs_force_ff_Newtonian_HuAdams_angular.F90:166-229: everything
      // along e = d / r
      const double du = DIM == 3 ? fma(d2, u2, fma(d1, u1, d0 * u0)) : fma(d1, u1, d0 * u0);
      const double aij = (bi + bj) * gw;
      double sc = P.eta_coef * P.eta * aij * du * (ir * ir) - aij * pij;
      if (P.noise) {
        const uint32_t pidj = pid_j();
        float g[4];
        pair_normals(P.seed, pidi < pidj ? pidi : pidj, pidi < pidj ? pidj : pidi, step, g);
        sc = sc + (double)g[0] * P.sqrt_2kt_eta * sqrt_nr(-P.eta_coef * aij * ir) * P.inv_sqrt_dt;
      }
      sc = sc * ir;
      a0 = sc * d0;
      a1 = sc * d1;
      a2 = sc * d2;
    } else {
      const double gir = gw * ir;
      const double fd = (COLL && FT >= 5 ? P.eta * bsum : fma(P.eta, bj, P.eta * bi)) * gir;
      if (FT == 3) {
        // rhs_force_ff_Newtonian_HuAdams.F90:140-237
        const double fcr = psum * gir;
        a0 = fd * u0 - fcr * d0;
        a1 = fd * u1 - fcr * d1;
        a2 = fd * u2 - fcr * d2;
      } else {
        // rhs_force_ff_non_Newtonian_HuAdams.F90:105-131 (FT 5; Espanol's,
        // FT 6, differs only in the noise; the angular form, FT 7, below) with
        // Pi = (p + G) I - G c (particles_compute_pressure_tensor.F90:114-133),
        // and the velocity gradient of pp_vgt_ip.inc:16-20
        const double dx[3] = {d0, d1, d2};
        // a boundary particle's gradient divides by its fluid partner's n
        const double gfac =
            COLL ? gir * ((cpair && sidi != 0) ? 1.0 / S.rho[j] : inv_ni) : gir;
        const double ug[3] = {-u0 * gfac, -u1 * gfac, -u2 * gfac};
#pragma unroll
        for (int b = 0; b < DIM; ++b)
#pragma unroll
          for (int a = 0; a < DIM; ++a) t[DIM + a + DIM * b] = ug[a] * dx[b];
        // j's Pi / n^2 (c is symmetric)
        const double pjb[9] = {rj.q0.x, rj.q1.y, rj.q2.x, rj.q1.y, rj.q0.y,
                               rj.q2.y, rj.q2.x, rj.q2.y, rj.q1.x};
        double fc[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int jj = 0; jj < DIM; ++jj)
#pragma unroll
          for (int a = 0; a < DIM; ++a) {
            const double ptjb = DIM == 3 ? pjb[a + 3 * jj] : pjb[(a == jj ? (a == 0 ? 0 : 4) : 1)];
            // colloid pairs: the fluid particle's Pi / n^2 on both sides
            const double ptib = FT == 7 ? pti[a + DIM * jj] * bi : pti[a + DIM * jj];
            double pij2 = cpair ? (sidi == 0 ? ptib + ptib : ptjb + ptjb) : ptib + ptjb;
            // rhs_force_ff_non_Newtonian_HuAdams_angular.F90: the diagonal
            // averaged, (Pi_i + Pi_j) / 2 (1/n_i^2 + 1/n_j^2)
            if (FT == 7 && a == jj) pij2 = 0.5 * (pti[a + DIM * jj] + ptjb / bj) * (bi + bj);
            fc[jj] = fc[jj] + pij2 * dx[a];
          }
        if (FT == 7) {
          // its dissipative term acts along e: eta_coef eta (1/n_i^2 +
          // 1/n_j^2) W' (e . v_ij) / r
          const double dv = DIM == 3 ? fma(d2, u2, fma(d1, u1, d0 * u0)) : fma(d1, u1, d0 * u0);
          const double fde = P.eta_coef * P.eta * (bi + bj) * gw * dv * (ir * ir * ir);
          a0 = fde * d0 - fc[0] * gir;
          a1 = fde * d1 - fc[1] * gir;
          a2 = DIM == 3 ? fde * d2 - fc[2] * gir : 0.0;
        } else {
          a0 = fd * u0 - fc[0] * gir;
          a1 = fd * u1 - fc[1] * gir;
          a2 = DIM == 3 ? fd * u2 - fc[2] * gir : 0.0;
        }
      }
      if (FT == 6 && P.noise) {
        espanol_noise(pid_j(), d0, d1, d2, ir,
                      gw * ir * inv_ni / S.rho[j], a0, a1, a2);
      } else if (FT != 7 && P.noise) {
        // f_r W e with W e = s ca (g + cb / ca (g.e) e), e = d / r, s = +1 when
        // pid_i < pid_j (noise_vector), written on d to save operations
        const uint32_t pidj = pid_j();
        float g[4];
        pair_normals(P.seed, pidi < pidj ? pidi : pidj, pidi < pidj ? pidj : pidi, step, g);
        // sqrt(-4 kT f_d / dt) / sqrt(2) as one root, in units of cg < 0 (the
        // unit turns the sign)
        const double fr = sqrt_pos(P.knoise * fd);
        const double sfr = pidi < pidj ? -fr : fr;
        const double g0 = (double)g[0], g1 = (double)g[1];
        if (DIM == 3) {
          // cb / ca
          const double cba = 0.81649658092772603273 * 1.41421356237309504880 - 1.0;
          const double g2 = (double)g[2];
          const double k = cba * fma(g2, d2, fma(g1, d1, g0 * d0)) * (ir * ir);
          a0 = fma(sfr, fma(k, d0, g0), a0);
          a1 = fma(sfr, fma(k, d1, g1), a1);
          a2 = fma(sfr, fma(k, d2, g2), a2);
        } else {
          a0 = fma(sfr, g0, a0);
          a1 = fma(sfr, g1, a1);
        }
      }
    }
    t[0] = a0;
    t[1] = a1;
    if (DIM == 3) t[2] = a2;
  }

  // Espanol's thermal force (rhs_force_ff_Newtonian_Espanol.F90:198-249,
  // rhs_force_ff_non_Newtonian_Espanol.F90): (A S e + B tr e) / sqrt(dt)
  // with S the symmetric traceless part of the pair's Gaussian dW and tr
  // its trace / num_dim, Z = 4 kT W' / (r n_i n_j) (gnn = W' / (r n_i n_j)).
  // S and tr are independent: S e is drawn as in the Hu-Adams body, oriented
  // by the lower pid, and tr is the pair block's fourth normal over
  // sqrt(num_dim), shared by both sides.
  __device__ __forceinline__ void espanol_noise(uint32_t pidj, double d0, double d1, double d2,
                                                double ir, double gnn, double& a0, double& a1,
                                                double& a2) const {
    float g[4];
    pair_normals(P.seed, pidi < pidj ? pidi : pidj, pidi < pidj ? pidj : pidi, step, g);
    const double zij = 4.0 * P.kt * gnn;
    const double ea = 5.0 * P.eta / 3.0, eb = (DIM + 2.0) * P.eta / 3.0;
    const double aij = sqrt_nr(-zij * ea) * P.inv_sqrt_dt;
    const double bij = sqrt_nr(-zij * DIM / 2.0 * (eb + ea * (2.0 / DIM - 1.0))) * P.inv_sqrt_dt;
    const double saij = pidi < pidj ? aij : -aij;
    const double ca = 0.70710678118654752440;
    const double g0 = (double)g[0], g1 = (double)g[1];
    const double btr = bij * (double)g[3] * (DIM == 3 ? 0.57735026918962576451 : ca) * ir;
    if (DIM == 3) {
      const double cb = 0.81649658092772603273 - 0.70710678118654752440;
      const double g2 = (double)g[2];
      const double k = cb * fma(g2, d2, fma(g1, d1, g0 * d0)) * (ir * ir);
      a0 = fma(saij, fma(k, d0, ca * g0), fma(btr, d0, a0));
      a1 = fma(saij, fma(k, d1, ca * g1), fma(btr, d1, a1));
      a2 = fma(saij, fma(k, d2, ca * g2), fma(btr, d2, a2));
    } else {
      a0 = fma(saij, ca * g0, fma(btr, d0, a0));
      a1 = fma(saij, ca * g1, fma(btr, d1, a1));
    }
  }

  // A fluid particle and a colloid boundary particle
  // (pp_interaction_fc.inc, pp_interaction_cf.inc): the boundary particle
  // moves at the no-slip velocity seen from the fluid particle and carries
  // the fluid particle's pressure (pb); its own number density stays.  The
  // no-slip velocity is formed in the boundary particle's frame, where the
  // fluid particle sits at r_xc + (x_f - x_c) and moves at its image
  // velocity, so both sides of the pair see the same relative velocity
  // u = v_i - v_j.
  __device__ __forceinline__ void colloid_substitute(int j, int sj, const RecF64& rj, double d0,
                                                     double d1, double d2, double jump, double& u0,
                                                     double& u1, double& u2, double& pb) const {
    double vc[3];
    if (sidi == 0) {
      const CollHot C = S.coll_hot[sj - 1];
      const double xj[3] = {rj.a.x, rj.a.y, DIM == 3 ? rj.b.x : 0.0};
      double rxc[3], vcoll[3];
      coll_nearest<DIM>(P, C, xj, le_t, rxc, vcoll);
      const double rxf[3] = {rxc[0] + d0, rxc[1] + d1, DIM == 3 ? rxc[2] + d2 : 0.0};
      const double vf[3] = {vi0 - jump, vi1, DIM == 3 ? vi2 : 0.0};
      coll_noslip<DIM>(P, C, rxc, vcoll, rxf, vf, vc);
      u0 = vf[0] - vc[0];
      u1 = vf[1] - vc[1];
      u2 = DIM == 3 ? vf[2] - vc[2] : 0.0;
      pb = pi;
    } else {
      const CollHot C = S.coll_hot[sidi - 1];
      const double rxf[3] = {rxc_i[0] - d0, rxc_i[1] - d1, DIM == 3 ? rxc_i[2] - d2 : 0.0};
      const double vf[3] = {P.le_g >= 0 ? rj.c.x + jump : rj.c.x, rj.c.y, DIM == 3 ? rj.d.x : 0.0};
      coll_noslip<DIM>(P, C, rxc_i, vcoll_i, rxf, vf, vc);
      u0 = vc[0] - vf[0];
      u1 = vc[1] - vf[1];
      u2 = DIM == 3 ? vc[2] - vf[2] : 0.0;
      pb = S.p[j];
    }
  }
};

template <int DIM, int FT, bool DECIDE = false, bool LEAVE = false>
struct ForceMixed {
  const DevParams& P;
  const DeviceState& S;
  const Home& h;
  float vi0, vi1, vi2, ai, bi, pi;
  uint32_t pidi;
  int64_t step;            // noise step (the context's marching step)
  // Oldroyd-B: own Pi / n^2 (xx, yy, zz, xy, xz, yz), 1 / n
  float pb[6];
  float inv_ni;
  uint4 own;               // Verlet lists: own fixed-point position
  // the acceleration's components, then the velocity gradient's: with
  // Verlet lists FP64 sums of the FP32 terms; per-step lists sum the
  // acceleration compensated in FP32
  static constexpr int kTerms = DIM + (FT >= 5 ? DIM * DIM : 0);
  std::conditional_t<DECIDE, WideF, KahanF> facc[DIM];
  WideF gacc[DIM * DIM];
  // the terms leave out the kernel gradient's factor but for the power of two
  // in the records, and the velocity gradient's 1 / n_i (finish_pairs)
  static constexpr bool kUnit = DECIDE && (FT == 3 || FT == 5);
  static constexpr bool kImages = false;
  // Verlet lists: the records of a lane's kWalk entries are gathered before
  // the first pair is evaluated
  static constexpr bool kBatched = DECIDE;
  static constexpr int kBatch = 2;
  static constexpr int kWalk = 2;
  __device__ __forceinline__ double sum(int c) const {
    return c < DIM ? facc[c < DIM ? c : 0].value() : gacc[c < DIM ? 0 : c - DIM].value();
  }
  // j's velocity and 1/n^2, p/n^2 (p for the angular form), pid, Oldroyd-B
  // Pi / n^2 (xx, yy, zz, xy, xz, yz), and the position: fixed-point (Verlet
  // lists) or cell-relative
  struct Rec {
    uint4 x;
    float4 v;
    float an;
    float4 q;
    float2 q2;
  };
  __device__ __forceinline__ Rec load_rec(uint32_t j) const {
    Rec r;
    r.an = 0.f;
    r.q = make_float4(0.f, 0.f, 0.f, 0.f);
    r.q2 = make_float2(0.f, 0.f);
    if (DECIDE) {
      r.x = load_at(S.xq, j);
      r.v = load_at(S.vr, j);
      if (FT < 5) r.an = load_at(S.an32, j);
      if (FT >= 5) {
        r.q = load_at(S.qr, j);
        r.q2 = load_at(reinterpret_cast<const float2*>(S.qr2), j);
      }
      return r;
    }
    r.v = S.vr[j];
    float4 x;
    if (FT >= 5) {
      x = load_xyz(S.xa + j);
      const float4 q = S.qr[j], q2 = S.qr2[j];
      r.x.w = __float_as_uint(r.v.w);
      r.v.w = q.x;
      r.q = make_float4(q.y, q.z, q.w, q2.x);
      r.q2 = make_float2(q2.y, q2.z);
    } else {
      x = S.qr[j];
      r.an = x.w;
      r.x.w = P.noise ? (uint32_t)S.pid[j] : 0u;
    }
    r.x.x = __float_as_uint(x.x);
    r.x.y = __float_as_uint(x.y);
    r.x.z = __float_as_uint(x.z);
    return r;
  }
  __device__ __forceinline__ Rec gather(uint32_t ent) const {
    return load_rec(ent & kIndexMask);
  }
  __device__ __forceinline__ void add(const float (&t)[kTerms]) {
#pragma unroll
    for (int c = 0; c < kTerms; ++c) {
      if (c < DIM)
        facc[c < DIM ? c : 0].add(t[c]);
      else
        gacc[c < DIM ? 0 : c - DIM].add(t[c]);
    }
  }
  __device__ __forceinline__ void body(uint32_t ent) {
    const uint32_t j = ent & kIndexMask;
    const Rec r = load_rec(j);
    const Offsets o = decode_code(ent >> kCodeShift);
    float d0, d1, d2, t[kTerms];
    rel_diff<DIM>(P, h,
                  make_float4(__uint_as_float(r.x.x), __uint_as_float(r.x.y),
                              __uint_as_float(r.x.z), 0.f),
                  o, d0, d1, d2);
    eval((int)j, r, d0, d1, d2, mixed_s2(d0, d1, d2), le_dvf(P, h, o), t);
    add(t);
  }
  // (Verlet candidates take no in / out decision: outside the cut-off the
  // kernel gradient is 0.  An empty slot holds the lane's own particle, moved
  // outside.)
  template <int NB>
  __device__ __forceinline__ void terms_f(const uint32_t (&e)[NB], const bool (&ok)[NB],
                                          Rec (&r)[NB], float (&t)[NB][kTerms]) const {
    float d[NB][3], r2[NB];
    uint64_t empty = 0;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      fixed_diff<DIM>(h, own, r[k].x, d[k][0], d[k][1], d[k][2]);
      r2[k] = mixed_s2(d[k][0], d[k][1], d[k][2]);
      empty |= __ballot(!ok[k]);
    }
    uint64_t out[NB] = {};
    if constexpr (LEAVE) {
#pragma unroll
      for (int k = 0; k < NB; ++k) out[k] = __ballot(!(ok[k] && r2[k] < (float)P.cut2));
    }
    if (__builtin_expect(empty != 0, 0)) {
#pragma unroll
      for (int k = 0; k < NB; ++k) r2[k] = ok[k] ? r2[k] : 4.f * P.cut2_hi_f32;
    }
#pragma unroll
    for (int k = 0; k < NB; ++k)
      eval((int)(e[k] & kIndexMask), r[k], d[k][0], d[k][1], d[k][2], r2[k], 0.f, t[k]);
    if constexpr (LEAVE) leave_out(out, t);
  }
  template <int NB>
  __device__ __forceinline__ void terms(const uint32_t (&e)[NB], const bool (&ok)[NB],
                                        Rec (&r)[NB], double (&t)[NB][kTerms]) const {
    float f[NB][kTerms];
    terms_f(e, ok, r, f);
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
      for (int c = 0; c < kTerms; ++c) t[k][c] = (double)f[k][c];
  }
  template <int NB>
  __device__ __forceinline__ void body_batch(const uint32_t (&e)[NB], const bool (&ok)[NB]) {
    float t[NB][kTerms];
    Rec r[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) r[k] = gather(e[k]);
    terms_f(e, ok, r, t);
#pragma unroll
    for (int k = 0; k < NB; ++k) add(t[k]);
  }
  // The terms of one pair: j's record, the separation and its square, the x
  // velocity of j's image on top of j's own.
  __device__ __forceinline__ void eval(int jidx, const Rec& rj, float d0, float d1, float d2,
                                       float r2, float jump, float (&t)[kTerms]) const {
    const float4& vj = rj.v;
    const float xjw = rj.an, bj = rj.v.w;
    const uint32_t pidj = rj.x.w;
    const float ir = __builtin_amdgcn_rsqf(r2);
    const float r = r2 * ir;
    float gw;
    if (kUnit) {
      gw = kernel_g_f32(P.kernel_type, r * P.inv_hf);
    } else {
      float w;
      kernel_w_gradw_f32(P.kernel_type, r * P.inv_hf, P.coeff, P.coef_gradf, w, gw);
    }
    const float u0 = vi0 - (DECIDE ? vj.x : vj.x + jump), u1 = vi1 - vj.y, u2 = vi2 - vj.z;
    float fi0, fi1, fi2;
    if (FT >= 5) {
      // rhs_force_ff_non_Newtonian_HuAdams.F90:105-131 with the records'
      // Pi / n^2, and the velocity gradient of pp_vgt_ip.inc:16-20 (FT 6,
      // Espanol: its thermal force below; FT 7, angular: the diagonal
      // averaged, (Pi_i + Pi_j) / 2 (1/n_i^2 + 1/n_j^2), and dissipation
      // along e)
      float sxx = pb[0] + rj.q.x, syy = pb[1] + rj.q.y, szz = pb[2] + rj.q.z;
      if (FT == 7) {
        const float bsum = bi + bj;
        sxx = 0.5f * (pb[0] / bi + rj.q.x / bj) * bsum;
        syy = 0.5f * (pb[1] / bi + rj.q.y / bj) * bsum;
        szz = 0.5f * (pb[2] / bi + rj.q.z / bj) * bsum;
      }
      const float sxy = pb[3] + rj.q.w, sxz = pb[4] + rj.q2.x, syz = pb[5] + rj.q2.y;
      float c0, c1, c2;
      if (DIM == 3) {
        c0 = sxx * d0 + sxy * d1 + sxz * d2;
        c1 = sxy * d0 + syy * d1 + syz * d2;
        c2 = sxz * d0 + syz * d1 + szz * d2;
      } else {
        c0 = sxx * d0 + sxy * d1;
        c1 = sxy * d0 + syy * d1;
        c2 = 0.f;
      }
      const float gir = gw * ir;
      const float f_d = P.etaf * (bi + bj) * gir;
      if (FT == 7) {
        const float fde = P.eta_coeff * P.etaf * (bi + bj) * gw * (d0 * u0 + d1 * u1 + d2 * u2) *
                          (ir * ir * ir);
        fi0 = fde * d0 - c0 * gir;
        fi1 = fde * d1 - c1 * gir;
        fi2 = fde * d2 - c2 * gir;
      } else {
        fi0 = f_d * u0 - c0 * gir;
        fi1 = f_d * u1 - c1 * gir;
        fi2 = f_d * u2 - c2 * gir;
      }
      const float gfac = kUnit ? gir : gir * inv_ni;
      const float ug[3] = {-u0 * gfac, -u1 * gfac, -u2 * gfac};
      const float dx[3] = {d0, d1, d2};
#pragma unroll
      for (int b = 0; b < DIM; ++b)
#pragma unroll
        for (int a = 0; a < DIM; ++a)
          t[DIM + a + DIM * b] = ug[a] * dx[b];
      if (FT == 6 && P.noise) {
        // Espanol's (A S e + B tr e) / sqrt(dt), Z = 4 kT W' / (r n_i n_j)
        float w0, w1, w2, g3;
        noise_vector<DIM, float>(P, step, pidi, pidj, d0 * ir, d1 * ir, d2 * ir, w0, w1, w2, &g3);
        const float zij = 4.0f * P.ktf * gir * inv_ni * __builtin_amdgcn_sqrtf(bj);
        const float ea = 5.0f * P.etaf / 3.0f, eb = (DIM + 2.0f) * P.etaf / 3.0f;
        const float aij = __builtin_amdgcn_sqrtf(-zij * ea) * P.inv_sqrt_dtf;
        const float bij = __builtin_amdgcn_sqrtf(-zij * DIM / 2.0f * (eb + ea * (2.0f / DIM - 1.0f))) *
                          P.inv_sqrt_dtf;
        const float btr = bij * g3 * (DIM == 3 ? 0.57735026918962576f : 0.70710678118654752f) * ir;
        fi0 = fi0 + aij * w0 + btr * d0;
        fi1 = fi1 + aij * w1 + btr * d1;
        fi2 = fi2 + aij * w2 + btr * d2;
      } else if (FT == 5 && P.noise) {
        if constexpr (kUnit) {
          unit_noise(pidj, f_d, d0, d1, d2, ir, fi0, fi1, fi2);
        } else {
        float w0, w1, w2;
        noise_vector<DIM, float>(P, step, pidi, pidj, d0 * ir, d1 * ir, d2 * ir, w0, w1, w2);
        const float f_r = __builtin_amdgcn_sqrtf(-4.0f * P.ktf * f_d) * P.inv_sqrt_dtf;
        fi0 = fi0 + f_r * w0;
        fi1 = fi1 + f_r * w1;
        fi2 = fi2 + f_r * w2;
        }
      }
    } else if (FT == 1) {
      // rhs_force_ff_Newtonian_Morris.F90:112-136 (accelerations carrying
      // the partner's mass; bi, vj.w = 1/rho)
      const float mj = (float)S.m[jidx];
      const float fcm = mj * (ai + xjw) * gw * ir;
      const float fdm = mj * 2.0f * P.etaf * gw * bi * bj * ir;
      fi0 = fdm * u0 - fcm * d0;
      fi1 = fdm * u1 - fcm * d1;
      fi2 = fdm * u2 - fcm * d2;
    } else if (FT == 2) {
      // rhs_force_ff_Newtonian_Espanol.F90:152-251 (bi, vj.w = 1/n)
      const float gnn = gw * bi * bj * ir;
      const float ev = (d0 * u0 + d1 * u1 + d2 * u2) * ir;
      const float fd1 = (2.0f - 1.0f / DIM) * P.etaf * gnn;
      const float fd2 = P.etaf * (DIM + 2.0f) / DIM * gnn * ev;
      const float se = (fd2 - (ai + xjw) * gw) * ir;
      fi0 = fd1 * u0 + se * d0;
      fi1 = fd1 * u1 + se * d1;
      fi2 = fd1 * u2 + se * d2;
      if (P.noise) {
        // (A S e + B tr e) / sqrt(dt), tr = g[3] / sqrt(num_dim)
        float w0, w1, w2, g3;
        noise_vector<DIM, float>(P, step, pidi, pidj, d0 * ir, d1 * ir, d2 * ir, w0, w1, w2, &g3);
        const float zij = 4.0f * P.ktf * gnn;
        const float ea = 5.0f * P.etaf / 3.0f, eb = (DIM + 2.0f) * P.etaf / 3.0f;
        const float aij = __builtin_amdgcn_sqrtf(-zij * ea) * P.inv_sqrt_dtf;
        const float bij = __builtin_amdgcn_sqrtf(-zij * DIM / 2.0f * (eb + ea * (2.0f / DIM - 1.0f))) *
                          P.inv_sqrt_dtf;
        const float btr = bij * g3 * (DIM == 3 ? 0.57735026918962576f : 0.70710678118654752f) * ir;
        fi0 = fi0 + aij * w0 + btr * d0;
        fi1 = fi1 + aij * w1 + btr * d1;
        fi2 = fi2 + aij * w2 + btr * d2;
      }
    } else if (FT == 3) {
      const float fcr = kUnit ? (ai + xjw) * (gw * ir) : (ai + xjw) * gw * ir;
      const float f_d = kUnit ? fmaf(P.etaf, bj, P.etaf * bi) * (gw * ir) : P.etaf * (bi + bj) * gw * ir;
      fi0 = f_d * u0 - fcr * d0;
      fi1 = f_d * u1 - fcr * d1;
      fi2 = f_d * u2 - fcr * d2;
      if (P.noise) {
        if constexpr (kUnit) {
          unit_noise(pidj, f_d, d0, d1, d2, ir, fi0, fi1, fi2);
        } else {
        float w0, w1, w2;
        noise_vector<DIM, float>(P, step, pidi, pidj, d0 * ir, d1 * ir, d2 * ir, w0, w1, w2);
        const float f_r = __builtin_amdgcn_sqrtf(-4.0f * P.ktf * f_d) * P.inv_sqrt_dtf;
        fi0 = fi0 + f_r * w0;
        fi1 = fi1 + f_r * w1;
        fi2 = fi2 + f_r * w2;
        }
      }
    } else {
      const float ev = (d0 * u0 + d1 * u1 + d2 * u2) * ir;
      const float pij = (pi + xjw) * 0.5f;
      const float aij = (bi + bj) * gw;
      const float f_c = aij * pij;
      const float f_d = P.eta_coeff * P.etaf * aij * ev * ir;
      float sc = f_d - f_c;
      if (P.noise) {
        float g[4];
        pair_normals(P.seed, pidi < pidj ? pidi : pidj, pidi < pidj ? pidj : pidi, step, g);
        sc = sc + g[0] * P.sqrt_2kt_etaf * __builtin_amdgcn_sqrtf(-P.eta_coeff * aij * ir) *
                      P.inv_sqrt_dtf;
      }
      sc = sc * ir;
      fi0 = sc * d0;
      fi1 = sc * d1;
      fi2 = sc * d2;
    }
    t[0] = fi0;
    t[1] = fi1;
    if (DIM == 3) t[2] = fi2;
  }
  // f_r W e of the Hu-Adams forms in units of the kernel gradient's factor
  // (negative: the unit turns the sign), as ForceF64 writes it on d
  __device__ __forceinline__ void unit_noise(uint32_t pidj, float f_d, float d0, float d1, float d2,
                                             float ir, float& f0, float& f1, float& f2) const {
    float g[4];
    pair_normals(P.seed, pidi < pidj ? pidi : pidj, pidi < pidj ? pidj : pidi, step, g);
    const float fr = __builtin_amdgcn_sqrtf(P.knoisef * f_d);
    const float sfr = pidi < pidj ? -fr : fr;
    if (DIM == 3) {
      const float cba = 0.81649658092772603273f * 1.41421356237309504880f - 1.0f;
      const float k = cba * fmaf(g[2], d2, fmaf(g[1], d1, g[0] * d0)) * (ir * ir);
      f0 = fmaf(sfr, fmaf(k, d0, g[0]), f0);
      f1 = fmaf(sfr, fmaf(k, d1, g[1]), f1);
      f2 = fmaf(sfr, fmaf(k, d2, g[2]), f2);
    } else {
      f0 = fmaf(sfr, g[0], f0);
      f1 = fmaf(sfr, g[1], f1);
    }
  }
};


template <int DIM>
__device__ __forceinline__ void finish_force(const DevParams& P, const DeviceState& S, int i,
                                             double f0, double f1, double f2,
                                             bool fluid = true) {
  const int64_t n = P.n;
  // fluid particles only (particles_apply_body_force.F90:173); the body
  // forces of types 2 and 3 follow in k_body_force
  if (P.body_force == 1 && fluid) {
    // particles_apply_body_force.F90:125-193
    if (fabs(P.bf[0]) > 1e-14) f0 = f0 + P.bf[0];
    if (fabs(P.bf[1]) > 1e-14) f1 = f1 + P.bf[1];
    if (DIM == 3 && fabs(P.bf[2]) > 1e-14) f2 = f2 + P.bf[2];
  }
  S.f[i] = f0;
  S.f[n + i] = f1;
  if (DIM == 3) S.f[2 * n + i] = f2;
}

// particles_compute_act.F90:140-155 on particle i's own ct and velocity
// gradient L: stores vgt = L and act = c L^T + L c - (c - I) / tau.
template <int DIM>
__device__ __forceinline__ void conformation_rate(const DevParams& P, const DeviceState& S, int i,
                                                  const double* L) {
  const int64_t n = P.n;
  const int d2n = DIM * DIM;
  double cc[9];
#pragma unroll
  for (int q = 0; q < d2n; ++q) {
    cc[q] = S.ct[(int64_t)q * n + i];
    S.vgt[(int64_t)q * n + i] = L[q];
  }
#pragma unroll
  for (int b = 0; b < DIM; ++b)
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      double t = 0.0;
#pragma unroll
      for (int k = 0; k < DIM; ++k)
        t = t + cc[a + DIM * k] * L[b + DIM * k] + L[a + DIM * k] * cc[k + DIM * b];
      double id = a == b ? 1.0 : 0.0;
      S.act[(int64_t)(a + DIM * b) * n + i] = t - (cc[a + DIM * b] - id) / P.tau;
    }
}

// The FP64 walk of per-step lists (without colloids) takes 8 KB of LDS per
// workgroup, its entry buffer plus a reserve.  That holds it to five waves
// per SIMD: each lane's gather touches a line of its own, and more waves take
// each other's lines from the L1.  (The 128^3 box: 1.99 ms per pass with six
// waves, 1.88 with five, before the noise's present form; 1.70 with five now,
// 1.75 with four.)  Oldroyd-B's records are 112 bytes: held below three waves,
// 100^3 1.56 ms instead of 1.60, 64^3 354 us instead of 367.
template <int FT>
constexpr int kForceLdsWordsF64 = FT >= 5 ? 4096 : 2048;

// What the pair bodies need of the home particle ii.
template <int DIM, int FT, bool DECIDE, bool LEAVE>
__device__ __forceinline__ ForceMixed<DIM, FT, DECIDE, LEAVE> mixed_policy(const DevParams& P,
                                                                           const DeviceState& S,
                                                                           const Home& h) {
  const int ii = h.ii;
  const float4 vi = S.vr[ii];
  const float4 qi = FT >= 5 || !DECIDE ? S.qr[ii] : make_float4(0.f, 0.f, 0.f, 0.f);
  ForceMixed<DIM, FT, DECIDE, LEAVE> pol{P, S, h, vi.x, vi.y, vi.z, 0.f, vi.w, 0.f,
                                         (uint32_t)S.pid[ii], S.step_dev[0]};
  if (FT <= 4) {
    // p/n^2, or p for the angular form
    const float an = DECIDE ? S.an32[ii] : qi.w;
    pol.ai = FT <= 3 ? an : 0.f;
    pol.pi = FT == 4 ? an : 0.f;
  } else if (DECIDE) {
    const float2 q2 = reinterpret_cast<const float2*>(S.qr2)[ii];
    pol.pb[0] = qi.x;
    pol.pb[1] = qi.y;
    pol.pb[2] = qi.z;
    pol.pb[3] = qi.w;
    pol.pb[4] = q2.x;
    pol.pb[5] = q2.y;
  } else {
    const float4 q2 = S.qr2[ii];
    pol.bi = qi.x;
    pol.pb[0] = qi.y;
    pol.pb[1] = qi.z;
    pol.pb[2] = qi.w;
    pol.pb[3] = q2.x;
    pol.pb[4] = q2.y;
    pol.pb[5] = q2.z;
  }
  if (FT >= 5) pol.inv_ni = (float)(1.0 / S.rho[ii]);
  if (DECIDE) pol.own = S.xq[ii];
  return pol;
}

template <int DIM, int FT, bool COLL, bool DECIDE, bool LEAVE>
__device__ __forceinline__ ForceF64<DIM, FT, COLL, DECIDE, LEAVE> f64_policy(const DevParams& P,
                                                                             const DeviceState& S,
                                                                             const Home& h) {
  const int ii = h.ii;
  const int64_t n = P.n;
  ForceF64<DIM, FT, COLL, DECIDE, LEAVE> pol{P, S, h};
  if (COLL) {
    pol.sidi = S.sid[ii];
    pol.le_t = S.time_dev[1];
    if (pol.sidi != 0) {
      const double xi[3] = {h.x0, h.x1, DIM == 3 ? h.x2 : 0.0};
      coll_nearest<DIM>(P, S.coll_hot[pol.sidi - 1], xi, pol.le_t, pol.rxc_i, pol.vcoll_i);
    }
  }
  pol.vi0 = S.v[ii];
  pol.vi1 = S.v[n + ii];
  pol.vi2 = DIM == 3 ? S.v[2 * n + ii] : 0.0;
  pol.ai = S.an[ii];
  pol.bi = S.bn[ii];
  pol.pi = S.p[ii];
  pol.inv_ni = 1.0 / S.rho[ii];
  pol.pidi = (uint32_t)S.pid[ii];
  pol.step = S.step_dev[0];
#pragma unroll
  for (int q = 0; q < pol.kTerms; ++q) pol.sum[q] = 0.0;
  if (FT >= 5) {
    // particles_compute_pressure_tensor.F90:114-133
#pragma unroll
    for (int b = 0; b < DIM; ++b)
#pragma unroll
      for (int a = 0; a < DIM; ++a) {
        double val = -P.G * S.ct[(int64_t)(a + DIM * b) * n + ii];
        if (a == b) val = val + pol.pi + P.G;
        pol.pti[a + DIM * b] = FT == 7 ? val : val * pol.bi;
      }
  }
  return pol;
}

// Acceleration (and conformation rate) of particle i from its pair sums, with
// the factors the bodies leave out: UNIT is that of the kernel gradient (0
// none, 1 FP64, 2 FP32 records), GRAD whether 1 / n_i is left out of the
// velocity gradient.
template <int DIM, int FT, int UNIT, bool GRAD>
__device__ __forceinline__ void finish_pairs(const DevParams& P, const DeviceState& S, int i,
                                             const double* sum, bool fluid) {
  const double unit = UNIT == 1 ? P.cg : (UNIT == 2 ? P.sum_scale : 1.0);
  // the Morris body sums accelerations already
  const double inv_mi = unit * (FT == 1 ? 1.0 : 1.0 / S.m[i]);
  finish_force<DIM>(P, S, i, sum[0] * inv_mi, sum[1] * inv_mi, DIM == 3 ? sum[DIM - 1] * inv_mi : 0.0,
                    fluid);
  if (FT >= 5) {
    // (the FP32 records' power of two scales the forces, not the gradient)
    const double fac = (UNIT == 2 ? unit * P.rec_scale : unit) * (GRAD ? 1.0 / S.rho[i] : 1.0);
    double L[DIM * DIM];
#pragma unroll
    for (int q = 0; q < DIM * DIM; ++q) L[q] = sum[DIM + q] * fac;
    conformation_rate<DIM>(P, S, i, L);
  }
}
template <int FT, bool MIXED, bool VERLET>
constexpr int kPairUnit = (FT == 3 || FT == 5) ? (MIXED ? (VERLET ? 2 : 0) : 1) : 0;
template <int FT, bool MIXED, bool COLL, bool VERLET>
constexpr bool kPairGrad = MIXED ? (VERLET && FT == 5) : !COLL;

// Whether the walk has left particles of a chunk to the scan: their forces (or
// velocity gradients) are not finite, and gate[4] says that there are some.
template <int DIM, int FT>
__device__ __forceinline__ bool lost_forces(const DeviceState& S, int64_t n, const Chunk& ch) {
  if (S.gate[4] == 0) return false;
  const int i = ch.p0 + (int)threadIdx.x;
  bool lost = false;
  if (i < ch.p1) {
    for (int d = 0; d < DIM; ++d) lost |= not_finite(S.f[d * n + i]);
    if (FT >= 5)
      for (int q = 0; q < DIM * DIM; ++q) lost |= not_finite(S.vgt[q * n + i]);
  }
  return __ballot(lost) != 0ull;
}

// One chunk slot of a force pass with one particle per lane.  Two launches
// over the same grid: SCAN = false takes the chunks whose lists hold every
// neighbour and walks them (per-step lists), SCAN = true takes the others
// and scans their stencil again; every chunk is done by exactly one launch.
// With colloids a box with sheared faces splits the chunks once more: the
// Lees-Edwards instantiation takes the rows within coll_le_cells of a face,
// the plain one (a quarter fewer registers) the interior.  VERLET: the scan
// takes the Verlet candidates, and the chunks whose walk left it particles
// (lost_forces).
template <int DIM, int FT, bool MIXED, bool COLL, bool LE, bool SCAN, bool VERLET>
__device__ __forceinline__ void forces_chunk(const DevParams& P, const DeviceState& S, int slot,
                                             int le_box, float4* __restrict__ tile,
                                             uint32_t* __restrict__ buf) {
  Chunk ch;
  if (!load_chunk(P, S, ch, slot)) return;
  if (SCAN && VERLET && !COLL) {
    if (!list_overflow(P, S, ch) && !lost_forces<DIM, FT>(S, P.n, ch)) return;
  } else if (list_overflow(P, S, ch) != SCAN) {
    return;
  }
  if (COLL && le_box >= 0 && chunk_meets_le_face(le_box, ch, P.coll_le_cells) != LE) return;
  const Home h = load_home<DIM>(P, S, ch);
  double sum[DIM + DIM * DIM];
  bool fluid = true;
  auto visit = [&](auto& pol) {
    if constexpr (SCAN) {
      int rechecks = 0;
      (void)staged_scan<DIM, std::remove_reference_t<decltype(pol)>, kTile, kBuf, VERLET>(
          P, S, ch, h, pol, tile, buf, rechecks, nullptr);
    } else {
      (void)tile;
      for_each_listed<DIM>(P, S, ch, h, pol, buf);
    }
  };
  if constexpr (MIXED) {
    auto pol = mixed_policy<DIM, FT, VERLET, SCAN && VERLET>(P, S, h);
    visit(pol);
#pragma unroll
    for (int c = 0; c < pol.kTerms; ++c) sum[c] = pol.sum(c);
  } else {
    auto pol = f64_policy<DIM, FT, COLL, VERLET, SCAN && VERLET>(P, S, h);
    visit(pol);
#pragma unroll
    for (int c = 0; c < pol.kTerms; ++c) sum[c] = pol.sum[c];
    fluid = !COLL || pol.sidi == 0;
  }
  if (h.active)
    finish_pairs<DIM, FT, kPairUnit<FT, MIXED, VERLET>, kPairGrad<FT, MIXED, COLL, VERLET>>(
        P, S, h.i, sum, fluid);
}

// With Verlet lists the rescan (SCAN) has work only if a list overflowed at
// the build or the walk has left it some; it is launched on a reduced grid,
// whose workgroups take every gridDim.x-th chunk slot, so that on the other
// steps its launch costs little.
template <int DIM, int FT, bool MIXED, bool COLL, bool LE, bool SCAN, bool VERLET = false>
__global__ __launch_bounds__(kWave) void k_forces(DevParams P, DeviceState S) {
  if (SCAN && VERLET && S.gate[2] == 0 && (COLL || S.gate[4] == 0)) return;
  const int le_box = P.le_g;
  if (!LE) P.le_g = -1;
  __shared__ float4 tile[SCAN ? kTile + 1 : 1];
  __shared__ uint32_t buf[(!MIXED && !COLL && !SCAN) ? kForceLdsWordsF64<FT> : kBuf * kWave];
  if (SCAN && VERLET) {
    const int slots = chunk_slots(P);
    for (int slot = blockIdx.x; slot < slots; slot += gridDim.x) {
      forces_chunk<DIM, FT, MIXED, COLL, LE, SCAN, VERLET>(P, S, slot, le_box, tile, buf);
      __syncthreads();
    }
  } else {
    forces_chunk<DIM, FT, MIXED, COLL, LE, SCAN, VERLET>(P, S, blockIdx.x, le_box, tile, buf);
  }
}

// The force walk of Verlet lists: 64 / LANES particles of a chunk per workgroup.
// SPEC: the quintic spline as a constant, with (kNoisy) or without (kQuiet)
// thermal noise, so that a batch's pairs form one block without run-time
// branches; kAny leaves both to the parameters.
enum ForceSpec { kAny = 0, kNoisy = 1, kQuiet = 2 };
//
// The FP64 Hu-Adams body is held to 128 registers, four waves per SIMD; left
// alone the compiler interleaves more of the two pairs' noise and takes 191.
// Two entries per lane and batch: the 128^3 box takes 1.33 ms with two, 1.47
// with four (191 registers); it took 1.66 with one particle per lane.  The
// mixed bodies fit six waves (0.87 ms, 1.14 with cell-relative positions, their
// code decode and compensated FP32 sums, one particle per lane).
//
// RESCAN (boxes with little more than a wave per SIMD, where registers cost
// nothing): a chunk whose lists overflowed is scanned again by its first
// workgroup, a wave whose sums are not finite walks its lists again, and
// k_forces is not launched (12^3 29.3 -> 27.9 us per step, 64 x 64 37.9 -> 36.4).
// The other boxes' walks leave such sums to k_forces: a second walk in them took
// registers (10 to 35, and with them a wave per SIMD).
template <int DIM, int FT, bool MIXED, bool COLL, bool LE, int SPEC, int LANES, bool RESCAN = false>
__global__ __launch_bounds__(kWave, RESCAN ? (SPEC == kQuiet && FT <= 4 ? 4 : 2) : ((!MIXED && !COLL && FT == 3) ? 4 : (MIXED ? (FT >= 5 && LANES == 16 ? 3 : 6) : 1))) void k_force_walk(DevParams P, DeviceState S) {
  const int le_box = P.le_g;
  if (!LE) P.le_g = -1;
  if (SPEC != kAny) {
    P.kernel_type = 1;
    P.noise = SPEC == kNoisy ? 1 : 0;
  }
  constexpr int kOwn = kPart<LANES>;
  int part;
  Chunk ch;
  const int slot = part_slot<LANES>(blockIdx.x, part);
  if (!load_chunk(P, S, ch, slot)) return;
  if (ch.p0 + kOwn * part >= ch.p1) return;
  if (COLL && le_box >= 0 && chunk_meets_le_face(le_box, ch, P.coll_le_cells) != LE) return;
  if (S.gate[2] != 0 && list_overflow(P, S, ch)) {
    if constexpr (RESCAN) {
      __shared__ float4 tile[kTile + 1];
      __shared__ uint32_t buf[kBuf * kWave];
      if (part == 0) forces_chunk<DIM, FT, MIXED, COLL, LE, true, true>(P, S, slot, le_box, tile, buf);
    }
    return;
  }
  const Home h = load_part_home<DIM, LANES>(P, S, ch, part);
  constexpr int kTerms = DIM + (FT >= 5 ? DIM * DIM : 0);
  __shared__ __align__(16) double lds[kTermWords<kTerms, LANES>];
  const int i = ch.p0 + kOwn * part + (int)threadIdx.x;
  const bool mine = threadIdx.x < kOwn && i < ch.p1;
  // true when a particle's sums are not finite
  auto pass = [&](auto leave) {
    constexpr bool kLeave = decltype(leave)::value;
    auto walk = [&](auto&& pol) { walk_part<DIM, LANES>(P, S, ch, part, h, pol, 0.0, lds); };
    if constexpr (MIXED)
      walk(mixed_policy<DIM, FT, true, kLeave>(P, S, h));
    else
      walk(f64_policy<DIM, FT, COLL, true, kLeave>(P, S, h));
    bool bad = false;
    if (mine) {
      double sum[kTerms];
#pragma unroll
      for (int c = 0; c < kTerms; ++c) {
        sum[c] = part_sum(lds, threadIdx.x, c);
        bad |= not_finite(sum[c]);
      }
      finish_pairs<DIM, FT, kPairUnit<FT, MIXED, true>, kPairGrad<FT, MIXED, COLL, true>>(
          P, S, i, sum, !COLL || S.sid[i] == 0);
    }
    return __ballot(bad) != 0ull;
  };
  const bool bad = pass(std::false_type{});
  if constexpr (!COLL) {
    if (__builtin_expect(bad, 0)) {
      if constexpr (RESCAN)
        (void)pass(std::true_type{});
      else if (threadIdx.x == 0)
        S.gate[4] = 1;  // every writer stores 1
    }
  }
}

// ---------------------------------------------------------------------
// neighbour-set signature: per particle, the number of in-cutoff
// neighbours and the wrapping sum of a hash of (pid_i, pid_j)
// ---------------------------------------------------------------------
__device__ __forceinline__ uint32_t pair_hash(uint32_t a, uint32_t b) {
  uint32_t h = a * 0x9E3779B1u ^ (b + 0x7F4A7C15u) * 0x85EBCA77u;
  h ^= h >> 15;
  h *= 0x2C1B3C6Du;
  h ^= h >> 12;
  return h;
}

// DECIDE (Verlet lists, between sorts): the scan takes every candidate
// within rc + skin and the body keeps the ones inside the cut-off on the
// current positions.
template <int DIM, bool DECIDE>
struct SignaturePol {
  const DevParams& P;
  const DeviceState& S;
  const Home& h;
  uint32_t pidi;
  uint32_t hs;
  int nin = 0;
  static constexpr bool kImages = true;
  static constexpr bool kBatched = false;
  __device__ __forceinline__ void body(uint32_t ent) {
    const int j = (int)(ent & kIndexMask);
    if (DECIDE) {
      const int64_t n = P.n;
      double d0, d1, d2;
      int sg;
      if (!(exact_d2_verlet<DIM>(P, h, S.x[j], S.x[n + j], DIM == 3 ? S.x[2 * n + j] : 0.0, d0,
                                 d1, d2, sg) < P.cut2))
        return;
    }
    ++nin;
    hs += pair_hash(pidi, (uint32_t)S.pid[j]);
  }
};

template <int DIM, bool LE, bool VERLET>
__global__ __launch_bounds__(kWave) void k_signature(DevParams P, DeviceState S) {
  if (!LE) P.le_g = -1;
  __shared__ float4 tile[kTile + 1];
  __shared__ uint32_t buf[kBuf * kWave];
  Chunk ch;
  if (!load_chunk(P, S, ch, blockIdx.x)) return;
  const Home h = load_home<DIM>(P, S, ch);
  SignaturePol<DIM, VERLET> pol{P, S, h, (uint32_t)S.pid[h.ii], 0u};
  int rechecks = 0;
  (void)staged_scan<DIM, SignaturePol<DIM, VERLET>, kTile, kBuf, VERLET>(P, S, ch, h, pol, tile,
                                                                         buf, rechecks, nullptr);
  if (!h.active) return;
  S.nbr_hash[h.i] = pol.hs;
  S.nbr_sig_count[h.i] = pol.nin;
  S.recheck[h.i] = rechecks;
}

// ---------------------------------------------------------------------
// launchers: one 64-lane workgroup per chunk; the grid covers the upper
// bound of chunks (one partial chunk per row plus n / 64 full ones)
// ---------------------------------------------------------------------
// Chunk slots from which a density walk takes a whole chunk per workgroup.
constexpr int kWholeChunkSlots = 4096;
// A box that leaves the 1024 SIMDs idle splits its work further.
// Sixteen lanes per particle while the four-lane walk has less than a wave per
// SIMD (density), three (forces); us per step with four lanes, and with sixteen
// in the density, in both: 12^3 47, 39, 28; 26^3 57, 56, 48 (30^3 with sixteen
// in the forces alone 50 instead of 59); 37 x 29 x 41 87, 91, 87 (84); 45^3 137,
// 146, 145; 128 x 128 52, 53, 52; Oldroyd-B 12^3 57, 49, 33, 26^3 71, 70, 61,
// 41^3 148, 154, 154.
constexpr int kWideDensity = 16 * 1024, kWideForces = 3 * 16 * 1024;
// Builds by four waves per chunk while a wave per chunk is less than one per
// SIMD; us per evaluation with one and with four: 12^3 177 and 129, 32^3 191
// and 170, mixed 175 and 161, 64 x 64 59 and 56; build and walk of 45^3 171
// and 209.
constexpr int kSplitSlots = 1024;

template <int DIM, bool MIXED, bool LE>
static void launch_density_walk(hipStream_t s, const DevParams& P, const DeviceState& S) {
  const int slots = chunk_slots(P);
  const dim3 b(kWave);
  const bool quintic = P.kernel_type == 1 && P.density_type == 2;
  if constexpr (!LE) {
    if (quintic && P.n < kWideDensity) {
      hipLaunchKernelGGL((k_density_walk<DIM, MIXED, LE, true, 1, 16>), dim3(16 * slots), b, 0, s,
                         P, S);
      return;
    }
  }
  // (the chunks next to sheared faces are few in any box: 64^3 with colloids 117
  // us with whole chunks, 57 with quarters)
  if (!LE && slots >= kWholeChunkSlots) {
    if (quintic)
      hipLaunchKernelGGL((k_density_walk<DIM, MIXED, false, true, 4, 4>), dim3(slots), b, 0, s, P, S);
    else
      hipLaunchKernelGGL((k_density_walk<DIM, MIXED, false, false, 4, 4>), dim3(slots), b, 0, s, P, S);
  } else {
    if (quintic)
      hipLaunchKernelGGL((k_density_walk<DIM, MIXED, LE, true, 1, 4>), dim3(4 * slots), b, 0, s, P,
                         S);
    else
      hipLaunchKernelGGL((k_density_walk<DIM, MIXED, LE, false, 1, 4>), dim3(4 * slots), b, 0, s, P,
                         S);
  }
}

// Workgroups of a launch that has work only after a list build or overflow (a
// multiple of 8, at most the slots): few enough that the launch is cheap on
// the other steps (on the 128^3 box, with 33k slots, two such launches cost
// 15 us less than with a workgroup per slot), and enough to fill the GPU.
static inline dim3 strided_grid(const DevParams& P) {
  return dim3(std::min(chunk_slots(P), 4096));
}

// Lists rebuilt every step, in the shape asked for.  (Verlet lists are built in
// the default one.  The build holds four waves per SIMD with either tile, and the
// larger one takes a row's records in one batch; a list buffer of 12 is the same
// ring of 16.  Density pass with a build, tiles of 224 and 128: 128^3 1.53 and
// 1.59 ms, 100^3 0.81 and 0.86, 45^3 150 and 184 us, Oldroyd-B 41^3 137 and 157,
// 256 x 256 36 and 37.)
template <int DIM, bool MIXED, bool LE>
static void launch_density_shape(hipStream_t s, const DevParams& P, const DeviceState& S) {
  const dim3 g(chunk_slots(P)), b(kWave);
  switch (P.density_shape) {
    case 1:
      hipLaunchKernelGGL((k_density<DIM, MIXED, 128, 16, LE, kStore>), g, b, 0, s, P, S);
      break;
    case 2:
      hipLaunchKernelGGL((k_density<DIM, MIXED, 224, 12, LE, kStore>), g, b, 0, s, P, S);
      break;
    case 3:
      hipLaunchKernelGGL((k_density<DIM, MIXED, 128, 12, LE, kStore>), g, b, 0, s, P, S);
      break;
    default:
      hipLaunchKernelGGL((k_density<DIM, MIXED, kTile, kBuf, LE, kStore>), g, b, 0, s, P, S);
  }
}

template <int DIM, bool MIXED>
static void launch_density_dim(hipStream_t s, const DevParams& P, const DeviceState& S) {
  if (!P.verlet) {
    if (P.le_g >= 0) launch_density_shape<DIM, MIXED, true>(s, P, S);
    launch_density_shape<DIM, MIXED, false>(s, P, S);
    return;
  }
  // Verlet lists: a box with sheared faces splits the chunks between
  // the Lees-Edwards and the plain instantiations, as its per-step lists do
  if constexpr (!MIXED) {  // mixed precision keeps per-step lists in sheared boxes
    if (P.le_g >= 0)
      hipLaunchKernelGGL((k_density<DIM, MIXED, kTile, kBuf, true, kScan>), strided_grid(P),
                         dim3(kWave), 0, s, P, S);
  }
  if (P.le_g < 0 && chunk_slots(P) < kSplitSlots)
    hipLaunchKernelGGL((k_density_split<DIM, MIXED>), strided_grid(P), dim3(kWave, 4), 0, s, P, S);
  else
    hipLaunchKernelGGL((k_density<DIM, MIXED, kTile, kBuf, false, kScan>), strided_grid(P),
                       dim3(kWave), 0, s, P, S);
  if constexpr (!MIXED) {
    if (P.le_g >= 0) launch_density_walk<DIM, MIXED, true>(s, P, S);
  }
  launch_density_walk<DIM, MIXED, false>(s, P, S);
}

void launch_density(hipStream_t s, const DevParams& P, const DeviceState& S, bool mixed) {
  if (P.dim == 3) {
    if (mixed)
      launch_density_dim<3, true>(s, P, S);
    else
      launch_density_dim<3, false>(s, P, S);
  } else {
    if (mixed)
      launch_density_dim<2, true>(s, P, S);
    else
      launch_density_dim<2, false>(s, P, S);
  }
}

void launch_eos(hipStream_t s, const DevParams& P, const DeviceState& S) {
  hipLaunchKernelGGL(k_eos, dim3((P.n + 255) / 256), dim3(256), 0, s, P, S);
}

void launch_refresh_records(hipStream_t s, const DevParams& P, const DeviceState& S) {
  hipLaunchKernelGGL(k_refresh_records, dim3((P.n + 255) / 256), dim3(256), 0, s, P, S);
}

template <int DIM, int FT, bool MIXED, bool COLL>
static void launch_forces_le(hipStream_t s, const DevParams& P, const DeviceState& S) {
  dim3 g(chunk_slots(P)), b(kWave);
  if (P.verlet) {
    // as the lists rebuilt every step: with colloids the chunks near a
    // sheared face take the Lees-Edwards instantiation and the others the
    // plain one; without, a sheared box runs the Lees-Edwards one alone
    const dim3 gq(4 * chunk_slots(P));
    if constexpr (!MIXED) {  // mixed precision keeps per-step lists in sheared boxes
      if (P.le_g >= 0) {
        hipLaunchKernelGGL((k_force_walk<DIM, FT, MIXED, COLL, true, kAny, 4>), gq, b, 0, s, P, S);
        hipLaunchKernelGGL((k_forces<DIM, FT, MIXED, COLL, true, true, true>), strided_grid(P), b,
                           0, s, P, S);
      }
    }
    if (P.le_g < 0 || COLL) {
      constexpr int kWithNoise = !COLL && FT != 1 && FT != 7 ? kNoisy : kAny;
      constexpr int kNoNoise = !COLL ? kQuiet : kAny;
      // (the common laws only: a variant of every law would double the library)
      constexpr bool kHasWide = !COLL && (FT == 3 || FT == 4 || FT == 5);
      const dim3 gw(16 * chunk_slots(P));
      if constexpr (kHasWide) {
        if (P.kernel_type == 1 && P.n < kWideDensity) {
          if (P.noise)
            hipLaunchKernelGGL((k_force_walk<DIM, FT, MIXED, COLL, false, kWithNoise, 16, true>), gw,
                               b, 0, s, P, S);
          else
            hipLaunchKernelGGL((k_force_walk<DIM, FT, MIXED, COLL, false, kNoNoise, 16, true>), gw,
                               b, 0, s, P, S);
          return;
        }
      }
      if (kHasWide && P.kernel_type == 1 && P.n <= kWideForces) {
        if constexpr (kHasWide) {
          if (P.noise)
            hipLaunchKernelGGL((k_force_walk<DIM, FT, MIXED, COLL, false, kWithNoise, 16>), gw, b,
                               0, s, P, S);
          else
            hipLaunchKernelGGL((k_force_walk<DIM, FT, MIXED, COLL, false, kNoNoise, 16>), gw, b, 0,
                               s, P, S);
        }
      } else if (P.kernel_type != 1)
        hipLaunchKernelGGL((k_force_walk<DIM, FT, MIXED, COLL, false, kAny, 4>), gq, b, 0, s, P, S);
      else if (P.noise)
        hipLaunchKernelGGL((k_force_walk<DIM, FT, MIXED, COLL, false, kWithNoise, 4>), gq, b, 0, s,
                           P, S);
      else
        hipLaunchKernelGGL((k_force_walk<DIM, FT, MIXED, COLL, false, kNoNoise, 4>), gq, b, 0, s, P,
                           S);
      hipLaunchKernelGGL((k_forces<DIM, FT, MIXED, COLL, false, true, true>), strided_grid(P), b,
                         0, s, P, S);
    }
    return;
  }
  if (P.le_g >= 0) {
    hipLaunchKernelGGL((k_forces<DIM, FT, MIXED, COLL, true, false>), g, b, 0, s, P, S);
    hipLaunchKernelGGL((k_forces<DIM, FT, MIXED, COLL, true, true>), g, b, 0, s, P, S);
  }
  if (P.le_g < 0 || COLL) {
    hipLaunchKernelGGL((k_forces<DIM, FT, MIXED, COLL, false, false>), g, b, 0, s, P, S);
    hipLaunchKernelGGL((k_forces<DIM, FT, MIXED, COLL, false, true>), g, b, 0, s, P, S);
  }
}

// Body forces that depend on the position (particles_apply_body_force.F90:
// 196-353), added to the accelerations of fluid particles after the force
// pass: type 2, +g_x below half of max_phys along the last dimension and
// -g_x above it (nothing on the line itself); type 3, g_x sin(k y) with
// k = 2 pi / (max_phys(2) - min_phys(2)).  Kept out of the pair kernels,
// whose registers the sine would otherwise take.
__global__ void k_body_force(DevParams P, DeviceState S) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  if (P.ncoll && S.sid[i] != 0) return;  // :246, :252, :330
  const int64_t n = P.n;
  double f0 = S.f[i];
  if (P.body_force == 2) {
    const double xl = S.x[(int64_t)(P.dim - 1) * n + i];
    if (xl < P.bf_split)
      f0 = f0 + P.bf[0];
    else if (xl > P.bf_split)
      f0 = f0 - P.bf[0];
  } else {
    f0 = f0 + P.bf[0] * sin(P.bf_k * S.x[n + i]);
  }
  S.f[i] = f0;
}

template <int DIM>
static void launch_forces_dim(hipStream_t s, const DevParams& P, const DeviceState& S,
                              bool mixed) {
  // Oldroyd-B: 5 Hu-Adams, 6 Espanol, 7 angular (rhs_force_ff_non_Newtonian.F90)
  const int ft = P.newtonian ? P.force_type : (P.force_type == 3 ? 5 : (P.force_type == 2 ? 6 : 7));
  if (mixed) {
    if (ft == 3)
      launch_forces_le<DIM, 3, true, false>(s, P, S);
    else if (ft == 4)
      launch_forces_le<DIM, 4, true, false>(s, P, S);
    else if (ft == 1)
      launch_forces_le<DIM, 1, true, false>(s, P, S);
    else if (ft == 2)
      launch_forces_le<DIM, 2, true, false>(s, P, S);
    else if (ft == 6)
      launch_forces_le<DIM, 6, true, false>(s, P, S);
    else if (ft == 7)
      launch_forces_le<DIM, 7, true, false>(s, P, S);
    else
      launch_forces_le<DIM, 5, true, false>(s, P, S);
  } else if (P.ncoll) {
    // colloids: FP64 only (checked by the API)
    if (ft == 3)
      launch_forces_le<DIM, 3, false, true>(s, P, S);
    else if (ft == 4)
      launch_forces_le<DIM, 4, false, true>(s, P, S);
    else if (ft == 1)
      launch_forces_le<DIM, 1, false, true>(s, P, S);
    else if (ft == 2)
      launch_forces_le<DIM, 2, false, true>(s, P, S);
    else
      launch_forces_le<DIM, 5, false, true>(s, P, S);
  } else {
    if (ft == 3)
      launch_forces_le<DIM, 3, false, false>(s, P, S);
    else if (ft == 4)
      launch_forces_le<DIM, 4, false, false>(s, P, S);
    else if (ft == 1)
      launch_forces_le<DIM, 1, false, false>(s, P, S);  // Morris (FP64 only)
    else if (ft == 2)
      launch_forces_le<DIM, 2, false, false>(s, P, S);  // Espanol (FP64 only)
    else if (ft == 6)
      launch_forces_le<DIM, 6, false, false>(s, P, S);  // Oldroyd-B Espanol (FP64 only)
    else if (ft == 7)
      launch_forces_le<DIM, 7, false, false>(s, P, S);  // Oldroyd-B angular (FP64 only)
    else
      launch_forces_le<DIM, 5, false, false>(s, P, S);
  }
}

void launch_forces(hipStream_t s, const DevParams& P, const DeviceState& S, bool mixed) {
  if (P.dim == 3)
    launch_forces_dim<3>(s, P, S, mixed);
  else
    launch_forces_dim<2>(s, P, S, mixed);
  if (P.body_force >= 2)
    hipLaunchKernelGGL(k_body_force, dim3((P.n + 255) / 256), dim3(256), 0, s, P, S);
}

void launch_signature(hipStream_t s, const DevParams& P, const DeviceState& S, bool mixed) {
  (void)mixed;  // both modes share the decision
  dim3 g(chunk_slots(P)), b(kWave);
  const bool le = P.le_g >= 0;
  if (P.dim == 3) {
    if (P.verlet && le)
      hipLaunchKernelGGL((k_signature<3, true, true>), g, b, 0, s, P, S);
    else if (P.verlet)
      hipLaunchKernelGGL((k_signature<3, false, true>), g, b, 0, s, P, S);
    else if (le)
      hipLaunchKernelGGL((k_signature<3, true, false>), g, b, 0, s, P, S);
    else
      hipLaunchKernelGGL((k_signature<3, false, false>), g, b, 0, s, P, S);
  } else {
    if (P.verlet && le)
      hipLaunchKernelGGL((k_signature<2, true, true>), g, b, 0, s, P, S);
    else if (P.verlet)
      hipLaunchKernelGGL((k_signature<2, false, true>), g, b, 0, s, P, S);
    else if (le)
      hipLaunchKernelGGL((k_signature<2, true, false>), g, b, 0, s, P, S);
    else
      hipLaunchKernelGGL((k_signature<2, false, false>), g, b, 0, s, P, S);
  }
}

}  // namespace sdpd
