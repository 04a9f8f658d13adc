// ghost_fill.h -- the ghost fill of one cell and the CFL time of one ghost
// cell, shared by the single-box kernels (kernels_common.hip) and the batched
// ones (kernels_batch.hip), so that a box's ghosts are filled bit for bit the
// same way in both.
//
// Reference correspondence (INL = library/mhd_solver.inl):
//   ghost_y_cell   communicate_gather_kernel_y + communicate_scatter_kernel_y
//                  (INL:90-286) with relative_displacement (INL:288-295)
//   ghost_z_cell   the Z halo copies of communicate() (INL:446-708)
#pragma once

#include "nmhd_kernels.h"

namespace nmhd {

// Value of field f that the fill gives cell (x, ghost row j of the lower or
// upper slab, z); not the first upper ghost By face, which it keeps.
template <bool Upper>
__device__ __forceinline__ float ghost_y_value(const Box &b, const FieldPtrs &W,
                                               const GhostShear &g, int f, int x, int j, int z) {
#pragma clang fp contract(off)
  const int nx = b.n[0], M = b.m[1];
  int i = x;
  if (b.shear_y) {
    i = Upper ? x - g.n - 1 : x + g.n;  // |n| < nx
    i = i < 0 ? i + nx : i;
    i = i < 0 ? i + nx : (i >= nx ? i - nx : i);
  }
  const int row = Upper ? M + j : b.n[1] - 2 * M + j;
  float v = W.f[f][addr(b, i, row, z)];
  if (b.shear_y) {
    // the second source cell (the reference's val_inc1 / val_dec1)
    const float v1 = b.fix_interp ? W.f[f][addr(b, i + 1 < nx ? i + 1 : 0, row, z)] : v;
    // (1-d)*v + d*v, exactly as the gather kernel writes it (INL:108-110);
    // with fix_interp (1-d)*v0 + d*v1 and d*v0 + (1-d)*v1
    v = Upper ? g.part * v + (1.0f - g.part) * v1 : (1.0f - g.part) * v + g.part * v1;
    if (f == 1) {
      const float relvel = -b.qshear * b.omega * b.local_ext[1];
      v = Upper ? v + relvel : v - relvel;
    }
  }
  return v;
}

// The fill of cell (x, j, z) of the lower or upper M-row slab.  The first
// upper ghost By face (the outer radial face) is kept.  Cfl: returns the
// cell's CFL time, its upper faces formed from the fill's sources (a
// neighbour's may not be written yet); else +inf.
template <bool Upper, bool Cfl>
__device__ __forceinline__ float ghost_y_fill(const Box &b, const FieldPtrs &W, const GhostShear &g,
                                              int x, int j, int z) {
  const int nx = b.n[0], ny = b.n[1], nz = b.n[2], M = b.m[1];
  const long a = addr(b, x, Upper ? ny - M + j : j, z);
  const bool kept = Upper && j == 0;
  float v[8];
  for (int f = 0; f < 8; ++f)
    v[f] = f == 6 && kept ? W.f[6][a] : ghost_y_value<Upper>(b, W, g, f, x, j, z);
  float t = __uint_as_float(0x7f800000u);
  if (Cfl) {
    const int x1 = x + 1 < nx ? x + 1 : 0, z1 = z + 1 < nz ? z + 1 : 0;
    float byh;  // the next row: in the slab, or the interior's first, or (wrapped) the array's
    if (j + 1 < M)
      byh = ghost_y_value<Upper>(b, W, g, 6, x, j + 1, z);
    else
      byh = Upper ? ghost_y_value<false>(b, W, g, 6, x, 0, z) : W.f[6][addr(b, x, M, z)];
    const float w[5] = {v[0], v[1], v[2], v[3], v[4]}, lo[3] = {v[5], v[6], v[7]};
    const float hi[3] = {ghost_y_value<Upper>(b, W, g, 5, x1, j, z), byh,
                         ghost_y_value<Upper>(b, W, g, 7, x, j, z1)};
    t = cfl_time(b, w, lo, hi);
  }
  for (int f = 0; f < 8; ++f)
    if (!(f == 6 && kept)) W.f[f][a] = v[f];
  return t;
}

// The Y ghost cells of a box, i in [0, nx * 2M * nz): lower slab, then upper.
__device__ __forceinline__ long ghost_y_count(const Box &b) {
  return (long)b.n[0] * 2 * b.m[1] * b.n[2];
}
template <bool Cfl>
__device__ __forceinline__ float ghost_y_cell(const Box &b, const FieldPtrs &W,
                                              const GhostShear &g, long i) {
  // 32-bit index arithmetic: a box holds fewer than 2^31 cells
  const unsigned slab = (unsigned)(b.n[0] * b.m[1]) * (unsigned)b.n[2];
  const bool upper = (unsigned)i >= slab;
  const unsigned u = (unsigned)i - (upper ? slab : 0u), line = u / (unsigned)b.n[0];
  const int x = (int)(u - line * (unsigned)b.n[0]);
  const int z = (int)(line / (unsigned)b.m[1]);
  const int j = (int)(line - (unsigned)z * (unsigned)b.m[1]);
  return upper ? ghost_y_fill<true, Cfl>(b, W, g, x, j, z)
               : ghost_y_fill<false, Cfl>(b, W, g, x, j, z);
}

// Z ghost planes, a in [0, nx * ny * M): [0, M) <- [nz-2M, nz-M),
// [nz-M, nz) <- [M, 2M).
__device__ __forceinline__ void ghost_z_cell(const Box &b, const FieldPtrs &W, long a) {
  const long unit = (long)b.n[0] * b.n[1] * b.m[2];
  for (int f = 0; f < 8; ++f) {
    float *p = W.f[f];
    p[a] = p[b.ncell - 2 * unit + a];
    p[b.ncell - unit + a] = p[unit + a];
  }
}

// Cells a ghost fill rewrites, for the CFL reduction: slab 0, the Y ghost
// rows (nx * 2My * nz cells); slab 1, the Z ghost planes plus the last
// interior plane, whose upper B_z face is a ghost face (nx * ny * (2Mz + 1)).
__device__ __forceinline__ long ghost_cfl_count(const Box &b, int slab) {
  const int M = slab == 0 ? b.m[1] : b.m[2];
  if (M == 0) return 0;
  return slab == 0 ? (long)b.n[0] * 2 * M * b.n[2] : (long)b.n[0] * b.n[1] * (2 * M + 1);
}

// CFL time of the i-th of those cells.
__device__ __forceinline__ float ghost_cfl_cell(const Box &b, const FieldPtrs &W, int slab,
                                                long i) {
  const int nx = b.n[0], ny = b.n[1], nz = b.n[2];
  const int M = slab == 0 ? b.m[1] : b.m[2];
  // 32-bit index arithmetic: a box holds fewer than 2^31 cells
  const unsigned u = (unsigned)i, row = u / (unsigned)nx;
  const int x = (int)(u - row * (unsigned)nx);
  int y, z;
  if (slab == 0) {
    const unsigned m2 = 2u * (unsigned)M;
    z = (int)(row / m2);
    const int r = (int)(row - (unsigned)z * m2);
    y = r < M ? r : ny - 2 * M + r;
  } else {
    const int r = (int)(row / (unsigned)ny);
    y = (int)(row - (unsigned)r * (unsigned)ny);
    z = r < M ? r : nz - 2 * M - 1 + r;
  }
  return cell_cfl(b, W, addr(b, x, y, z), x, y, z);
}

}  // namespace nmhd
