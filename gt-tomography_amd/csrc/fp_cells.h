// When the forward projector builds its packed volume copy (k_pack_cells), and how
// large it is.  Shared with the reconstruction server, which charges a request for it.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>

#include "cbct.h"

// z-fastest padded length: nz + 3 rounded up to 16 elements
inline size_t fp_zpadded(int nz) { return ((size_t)nz + 3 + 15) & ~size_t(15); }

// Upper bound on a view's detector rows with rays that leave through the volume's
// top or bottom: those that reach past its height at its far side (`off`: the
// view's v offset).
inline double fp_clipped_rows(const cbct_geom *g, double off) {
  const double R = 0.5 * std::sqrt((double)g->lx * g->lx + (double)g->ly * g->ly);
  const double vmax = 0.5 * g->lz * g->sdd / ((double)g->sad + R);   // heights up to here are never clipped
  const double pitch = (double)g->fov_v / g->nv;
  return std::max(0.0, 0.5 * g->fov_v + off - vmax) / pitch + std::max(0.0, 0.5 * g->fov_v - off - vmax) / pitch;
}

// Bytes of the packed copy for a projection with `rows` such rows over its views
// and n samples per ray, working copies of esz bytes; 0: none.  It is built
// when the clipped rays' samples outweigh building it: it costs 20 bytes of
// traffic per voxel (4.4 ps), the packed loads save about 1.6 ps a sample.  It
// must stay within a buffer's 4 GB.
inline size_t fp_cells_bytes(const cbct_geom *g, double rows, int n, size_t esz) {
  const size_t bytes = 4 * esz * fp_zpadded(g->nz) * ((size_t)g->nx + 3) * ((size_t)g->ny + 3);
  if (bytes >= (1ull << 32) - 64) return 0;
  const double nvox = (double)g->nx * g->ny * g->nz;
  return rows * g->nu * n > 3.6 * nvox ? bytes : 0;
}
