// sdpd_window.h -- the sheared window of a particle (host and device).
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define SDPD_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define SDPD_HOST_DEVICE inline
#endif

namespace sdpd {

// Cell of the frame shifted by sp (0 <= sp < the edge) that holds a particle of
// cell cx at xw, cells of edge cs.  A particle whose position is lost (not finite,
// or far outside the box after the run diverged) sits nowhere near its cell cx,
// which the sort clamped to the box; its window is its cell's, so that a wave's
// windows span at most its cells and three more and its stencil rows stay within
// three periods (RowPieces).  Between builds a particle is at most a quarter of a
// cell outside its own (half the largest skin).
SDPD_HOST_DEVICE int window_cell(double xw, int cx, double cs, double sp) {
  const double off = xw - (double)cx * cs;
  if (!(off > -0.5 * cs && off < 1.5 * cs)) xw = ((double)cx + 0.5) * cs;
  return (int)std::floor((xw - sp) / cs);
}

}  // namespace sdpd
