// tile_params.h -- the parameters of one launch of a tile kernel: the tracks, the
// spectral grid, the outputs and how they are cut into tiles.
#pragma once

#include "common.h"

namespace sr {

struct KParams {
  // tracks (CSR); offsets == nullptr selects the single-particle form
  const int64_t *offsets;
  const double *x, *y, *z, *ux, *uy, *uz;
  const double *weight;
  const uint32_t *it_start, *it_end, *it_snaps;
  uint32_t n_snaps, snaps_stride;
  double dt;
  int64_t single_n;
  double single_w;
  uint32_t single_its, single_ite;
  // grid
  int32_t comp;
  uint32_t n_omega, n_theta, n_phi;
  const double *omega, *sin_t, *cos_t, *radius, *sin_p, *cos_p;
  const double *screen_y;   // near, Cartesian screen: P = (radius[i], screen_y[j], L)
  double l_screen;
  double omega_step;        // rec sweep: omega[i+1] - omega[i]
  const double *form_factor;
  int64_t n_grid;
  // outputs (slices > 1: scratch[q][c] replaces out[c])
  int32_t n_out;
  double *out[kMaxOut];
  double *scratch;
  // 1: one snapshot and one output -- each thread sums its points over the
  // block's particles in LDS and adds the sum to the output once
  int32_t acc_lds;
  // per-particle outputs (the adjoint's fields): particle ip writes at
  // (ip - part_base) * part_stride past the usual index; 0 otherwise
  int64_t part_base, part_stride;
  // direction-independent step data from k_step_prep, or nullptr (the stage
  // then computes it), one record per sample: far [n_points][a_x, a_y, a_z,
  // bbar_x, bbar_y, bbar_z] (48 B, 16-byte aligned), near [n_points][b_x, b_y,
  // b_z].  One base address and fixed offsets: the stage reads a record with
  // three 16-byte loads and keeps no per-array base registers
  const double *pre;
  int64_t n_points;
  // tiling
  uint32_t n_chunks;
  uint32_t n_dir;
  UDiv div_chunks, div_dir, div_theta;   // by n_chunks, n_dir, n_theta (tiles < 2^31)
  int32_t slices;
  // tile kernel, FP64: the block's groups of threads that share a tile, each
  // sweeping a contiguous part of every track
  int32_t parts;
  int64_t n_tiles;
  int64_t slice_lo[kMaxSlices + 1];
  // launch order of the tiles (heaviest first), or nullptr: index order
  const int32_t *tile_order;
};

}  // namespace sr
