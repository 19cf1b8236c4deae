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
// when the clipped rays' samples outweigh building it: with FP32 copies it costs 20
// bytes of traffic per voxel (4.4 ps), the packed loads save about 1.6 ps a
// sample: 2.8 samples per voxel, and a second launch.  Both sides measured on slabs
// of 96^2 x 48 to 400^2 x 240: from 16 views on, 5 to 490 such samples per voxel, a
// projection with the copy takes 0.64 to 1.00 of the time without (FP32; 1.07 for
// 128^2 x 64, 16 views) and 0.53 to 1.01 (BF16, whose copy is half the bytes).  Fewer
// views gain or lose by their angles: 0.73 to 1.48 and 0.60 to 1.23.  It must stay
// within a buffer's 4 GB.
inline size_t fp_cells_bytes(const cbct_geom *g, double rows, int n, size_t esz) {
  const size_t bytes = 4 * esz * fp_zpadded(g->nz) * ((size_t)g->nx + 3) * ((size_t)g->ny + 3);
  if (bytes >= (1ull << 32) - 64) return 0;
  const double nvox = (double)g->nx * g->ny * g->nz;
  return rows * g->nu * n > 3.6 * nvox ? bytes : 0;
}
