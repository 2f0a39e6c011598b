// Device helpers shared by the ray kernels (render and gradient).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace at3d {

// LOCATE_GRID_CELL (shdomsub2.f:4043-4206) for a base grid without a tree.
__device__ inline int locate_cell_ray(const RayArgs& a, double& x0, double& y0, double z0) {
  const float* XG = a.xgrid;
  const float* YG = a.ygrid;
  const float* ZG = a.zgrid;
  if (!a.open_x) {
    const double xd = (double)(XG[a.nx] - XG[0]);
    if (x0 < XG[0])
      x0 = x0 - xd * (double)((int)((x0 - XG[0]) / xd) - 1);
    else if (x0 > XG[a.nx])
      x0 = x0 - xd * (double)(int)((x0 - XG[0]) / xd);
  }
  if (!a.open_y) {
    const double yd = (double)(YG[a.ny] - YG[0]);
    if (y0 < YG[0])
      y0 = y0 - yd * (double)((int)((y0 - YG[0]) / yd) - 1);
    else if (y0 > YG[a.ny])
      y0 = y0 - yd * (double)(int)((y0 - YG[0]) / yd);
  }
  int il = 0, iu = a.nx + 1;
  while (iu - il > 1) {
    const int im = (iu + il) / 2;
    if (x0 >= XG[im - 1]) il = im; else iu = im;
  }
  int ix = max(il, 1);
  il = 0;
  iu = a.ny + 1;
  while (iu - il > 1) {
    const int im = (iu + il) / 2;
    if (y0 >= YG[im - 1]) il = im; else iu = im;
  }
  int iy = max(il, 1);
  il = 0;
  iu = a.nz;
  while (iu - il > 1) {
    const int im = (iu + il) / 2;
    if (z0 >= ZG[im - 1]) il = im; else iu = im;
  }
  const int iz = max(il, 1);
  if (a.open_x) {
    if (x0 < XG[0]) ix = 1;
    else if (x0 > XG[a.nx - 1]) ix = a.nx + 1;
    else ix = ix + 1;
  }
  if (a.open_y) {
    if (y0 < YG[0]) iy = 1;
    else if (y0 > YG[a.ny - 1]) iy = a.ny + 1;
    else iy = iy + 1;
  }
  return (iz + (a.nz - 1) * (iy - 1) + (a.nz - 1) * a.nyc * (ix - 1)) - 1;
}

// One cell of a ray's path: corner points, box and flags.  REG: a base grid,
// where they follow from the cell's indices without loads that wait for one
// another (INIT_CELL_STRUCTURE shdomsub2.f:84-164: an open boundary's outer
// cells have no width); otherwise (a refined grid) from the cell arrays.
struct RayCell {
  int cell;          // -1: outside
  int ix, iy, iz;    // REG
  int gp[8];
  float lo[3], hi[3];
  int8_t fl;
};

template <bool REG>
__device__ inline void load_ray_cell(const RayArgs& a, RayCell& c) {
  if constexpr (REG) {
    const int x0 = a.open_x ? max(0, c.ix - 1) : c.ix, x1 = a.open_x ? min(a.nx - 1, c.ix) : c.ix + 1;
    const int y0 = a.open_y ? max(0, c.iy - 1) : c.iy, y1 = a.open_y ? min(a.ny - 1, c.iy) : c.iy + 1;
    const int sx = (x1 - x0) * a.ny1 * a.nz, sy = (y1 - y0) * a.nz;
    const int q = c.iz + a.nz * (y0 + a.ny1 * x0);
#pragma unroll
    for (int k = 0; k < 8; k++) c.gp[k] = q + ((k & 1) ? sx : 0) + ((k & 2) ? sy : 0) + (k >> 2);
    c.lo[0] = a.xgrid[x0];
    c.hi[0] = a.xgrid[x1];
    c.lo[1] = a.ygrid[y0];
    c.hi[1] = a.ygrid[y1];
    c.lo[2] = a.zgrid[c.iz];
    c.hi[2] = a.zgrid[c.iz + 1];
    c.fl = (int8_t)((a.open_x && (c.ix == 0 || c.ix == a.nx) ? 1 : 0) | (a.open_y && (c.iy == 0 || c.iy == a.ny) ? 2 : 0));
  } else {
    const int* gp = a.g.gridptr + (size_t)c.cell * 8;
#pragma unroll
    for (int k = 0; k < 8; k++) c.gp[k] = gp[k];
    const float* P = a.g.gridpos;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      c.lo[k] = P[c.gp[0] * 3 + k];
      c.hi[k] = P[c.gp[7] * 3 + k];
    }
    c.fl = a.g.cellflags[c.cell];
  }
}

// The cell a ray starts in.
template <bool REG>
__device__ inline void first_ray_cell(const RayArgs& a, int cell, RayCell& c) {
  c.cell = cell;
  if constexpr (REG) {
    const int nzc = a.nz - 1, t = cell / nzc;
    c.iz = cell - t * nzc;
    c.ix = t / a.nyc;
    c.iy = t - c.ix * a.nyc;
  }
  load_ray_cell<REG>(a, c);
}

// REG: the neighbour across the face a ray leaves by (its direction's face of
// dimension jface = 1, 2, 3), cell -1 beyond the bottom or top.  Rays leave an
// open side's outer cells by their inner faces only.
__device__ inline void next_ray_cell(const RayArgs& a, const RayCell& c, int jface, int bitx, int bity, int bitz,
                                     RayCell& n) {
  n.ix = c.ix;
  n.iy = c.iy;
  n.iz = c.iz;
  if (jface == 1) {
    n.ix += bitx ? -1 : 1;
    if (!a.open_x) n.ix = n.ix < 0 ? a.nx - 1 : n.ix == a.nx ? 0 : n.ix;
  } else if (jface == 2) {
    n.iy += bity ? -1 : 1;
    if (!a.open_y) n.iy = n.iy < 0 ? a.ny - 1 : n.iy == a.ny ? 0 : n.iy;
  } else {
    n.iz += bitz ? -1 : 1;
  }
  const int nxc = a.open_x ? a.nx + 1 : a.nx;
  const bool in = n.iz >= 0 && n.iz < a.nz - 1 && n.ix >= 0 && n.ix < nxc && n.iy >= 0 && n.iy < a.nyc;
  n.cell = in ? n.iz + (a.nz - 1) * (n.iy + a.nyc * n.ix) : -1;
}

}  // namespace at3d
