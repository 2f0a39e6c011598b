// Radiance rendering: one ray per lane (RENDER shdomsub4.f:93-286 with
// INTEGRATE_1RAY shdomsub2.f:2311-2743).
//
// The direction-dependent source at the grid points,
// COMPUTE_SOURCE_1CELL_UNPOL (shdomsub2.f:3046-3192) =
//   ext * ( sum_J S_J Y_J(dir)                       [spherical-harmonic source]
//           - sum_{l<=LS} T_l sum_{J in l} Y_J(dir) Ysun_J   [truncated single scatter]
//           + sum_pairs c * P_table(Theta) )          [exact single scatter, TMS]
// is computed once per distinct ray direction for every grid point (an MFMA
// product [points x nlm] x [nlm x directions] plus a per-point epilogue), so
// the ray kernel only gathers cell corners and integrates.
#include <hip/hip_runtime.h>
#include <math.h>

#include "kernels.h"
#include "ray_common.h"

namespace at3d {

__device__ inline int nterms_l(int l, int mm) {
  return (l <= mm) ? l * (l + 1) + l + 1 : (2 * mm + 1) * l - mm * mm + mm + 1;
}

// dsrc[p][d] = ext[p] * (raw[p][d] - sum_{l<=LS(p)} T[p][l] G[d][l] + sum_pairs c * ss[d][iph])
__global__ void k_dir_source_finish(const float* raw, int ldd, int ndir,
                                    const float* __restrict__ ext, const int* __restrict__ ns,
                                    const int* __restrict__ lofj, const float* __restrict__ tms,
                                    const float* __restrict__ G, const int32_t* __restrict__ ss_off,
                                    const int32_t* __restrict__ ss_iph,
                                    const float* __restrict__ ss_coef, const float* __restrict__ ssd,
                                    int numphase, int ml, int npts, int single_scatter, int tms_on,
                                    float* dsrc) {
  // raw and dsrc may be the same buffer: each element is read and then
  // written by one thread.
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npts * ndir) return;
  const int p = i / ndir, d = i - p * ndir;
  float v = single_scatter ? 0.0f : raw[(size_t)p * ldd + d];
  if (tms_on) {
    const int nsp = ns[p];
    if (!single_scatter && nsp > 0) {
      const int ls = lofj[nsp - 1];
      for (int l = 0; l <= ls; l++) v = v - tms[(size_t)p * (ml + 1) + l] * G[d * (ml + 1) + l];
    }
    for (int q = ss_off[p]; q < ss_off[p + 1]; q++) v = v + ss_coef[q] * ssd[d * numphase + ss_iph[q]];
  }
  dsrc[(size_t)p * ldd + d] = v * ext[p];
}



// The polarized direction source (COMPUTE_SOURCE_1CELL, shdomsub2.f:2868-3043)
// for I, Q and U: each block's spherical-harmonic sum less its truncated
// single scatter (a1 for I, b1 for Q and U, with their direction factors) plus
// the exact single scatter of the tabulated I, rotated Q and U.
__global__ void k_dir_source_finish_pol(const float* raw, int ldd, int cst, int ndir,
                                        const float* __restrict__ ext, const int* __restrict__ ns,
                                        const int* __restrict__ lofj, const float* __restrict__ tms,
                                        const float* __restrict__ tms5, const float* __restrict__ G3,
                                        const int32_t* __restrict__ ss_off, const int32_t* __restrict__ ss_iph,
                                        const float* __restrict__ ss_coef, const float* __restrict__ ssd,
                                        const float* __restrict__ ssq, const float* __restrict__ ssu,
                                        int numphase, int ml, int npts, int single_scatter, int tms_on,
                                        float* dsrc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npts * ndir) return;
  const int p = i / ndir, d = i - p * ndir;
  const size_t row = (size_t)p * ldd;
  float v[3];
  for (int k = 0; k < 3; k++) v[k] = single_scatter ? 0.0f : raw[row + k * cst + d];
  if (tms_on) {
    const int nsp = ns[p];
    if (!single_scatter && nsp > 0) {
      const int ls = lofj[nsp - 1];
      const size_t gd = (size_t)ndir * (ml + 1);
      for (int l = 0; l <= ls; l++) {
        const float t1 = tms[(size_t)p * (ml + 1) + l], t5 = tms5[(size_t)p * (ml + 1) + l];
        v[0] = v[0] - t1 * G3[d * (ml + 1) + l];
        v[1] = v[1] - t5 * G3[gd + d * (ml + 1) + l];
        v[2] = v[2] - t5 * G3[2 * gd + d * (ml + 1) + l];
      }
    }
    for (int q = ss_off[p]; q < ss_off[p + 1]; q++) {
      const float c = ss_coef[q];
      const int t = d * numphase + ss_iph[q];
      v[0] = v[0] + c * ssd[t];
      v[1] = v[1] + c * ssq[t];
      v[2] = v[2] + c * ssu[t];
    }
  }
  for (int k = 0; k < 3; k++) dsrc[row + k * cst + d] = v[k] * ext[p];
}

__device__ inline float trilin(const float* v8, double u, double v, double w) {
#pragma clang fp contract(off)
  return (float)((1 - w) * ((1 - v) * ((1 - u) * v8[0] + u * v8[1]) + v * ((1 - u) * v8[2] + u * v8[3])) +
                 w * ((1 - v) * ((1 - u) * v8[4] + u * v8[5]) + v * ((1 - u) * v8[6] + u * v8[7])));
}

// NST = 3: I, Q and U integrated along the ray with the same transmission;
// only I's source is clamped at zero, and Q and U have zero boundary
// radiances (the sky is unpolarized, the Lambertian surface depolarizes).
// REG (a base grid): the cells follow from their indices, and the next cell's
// eight extinctions and sources load while a cell is integrated; a wavefront
// has little beside it to hide a load behind (36864 rays are 576 of them), and
// the cell arrays made three loads wait for one another at every step: 9 views of
// 64 x 64 over 64 x 64 x 40 points 0.50 ms before, 0.37 now, one camera of 61 x 61
// 0.63 and 0.29.
// NST = 0: no radiances; the points around the cells the ray crosses go to its
// list (those the cell before did not have: four a step), for a call whose
// source is made at these points alone.  The path ends where the render's does,
// or (the gradient's traversal weighs the same extinctions in another order)
// a little past the end it is given in a.transcut.
template <int NST, bool REG>
__device__ inline void render_ray(const RayArgs& a, const PairArgs* pl, int ir) {
#pragma clang fp contract(off)
  constexpr int NS = NST > 0 ? NST : 1;
  int listed = 0;
  const double PI = acos(-1.0);
  const float* ZG = a.zgrid;
  const float* P = a.g.gridpos;
  double x0 = a.camx[ir], y0 = a.camy[ir], z0 = a.camz[ir];
  const double mu2 = a.cammu[ir], phi2 = a.camphi[ir];
  const double muray = -mu2, phiray = phi2 - PI;
  // extrapolate a sensor above the domain to the top (RENDER :223-236)
  if (z0 > (double)ZG[a.nz - 1]) {
    if (muray >= 0.0) {
      if constexpr (NST == 0) pl->cnt[ir] = 0;
      for (int k = 0; k < NST; k++) a.out[(size_t)ir * NST + k] = 0.0f;
      return;
    }
    const double r = ((double)ZG[a.nz - 1] - z0) / muray;
    x0 = x0 + r * sqrt(1 - muray * muray) * cos(phiray);
    y0 = y0 + r * sqrt(1 - muray * muray) * sin(phiray);
    z0 = ZG[a.nz - 1];
  }
  const int d = a.dir_of_ray[ir];
  const float topv = mu2 < 0.0 ? a.skyrad : 0.0f;
  const float* dsrc = a.dsrc + d * a.ds;
  const size_t LD = a.ps;
  const double eps = (double)(1.0e-5f * (P[a.g.gridptr[7] * 3 + 2] - P[a.g.gridptr[0] * 3 + 2]));
  const int maxcross = 500 * max(a.nx, max(a.ny, a.nz));
  double cx = sqrt(1.0 - mu2 * mu2) * cos(phi2 - PI);
  double cy = sqrt(1.0 - mu2 * mu2) * sin(phi2 - PI);
  double cz = -mu2, cxinv, cyinv, czinv;
  if (fabs(cx) > (double)1.0e-6f) cxinv = 1.0 / cx; else { cx = 0.0; cxinv = 1.0e6; }
  if (fabs(cy) > (double)1.0e-6f) cyinv = 1.0 / cy; else { cy = 0.0; cyinv = 1.0e6; }
  if (fabs(cz) > (double)1.0e-6f) czinv = 1.0 / cz; else { cz = 0.0; czinv = 1.0e6; }
  const int bitx = cx < 0.0, bity = cy < 0.0, bitz = cz < 0.0;
  const int ioct = bitx + 2 * bity + 4 * bitz;
  const float xm = 0.5f * (a.xgrid[0] + a.xgrid[a.nx - 1]);
  const float ym = 0.5f * (a.ygrid[0] + a.ygrid[a.ny - 1]);
  double xe = x0, ye = y0, ze = z0;
  const int start = [&] {
    const int c = locate_cell_ray(a, xe, ye, ze);   // (wraps xe, ye into a periodic domain)
    return !REG && c >= 0 && c < a.g.ncells ? locate_in_tree(a.g, c, xe, ye, ze) : c;
  }();
  if (start < 0 || start >= a.g.ncells) {
    if constexpr (NST == 0) pl->cnt[ir] = 0;
    else atomicOr(a.errflag, 4);
    for (int k = 0; k < NST; k++) a.out[(size_t)ir * NST + k] = 0.0f;
    return;
  }
  double radiance[NS], transmit = 1.0;
  for (int k = 0; k < NST; k++) radiance[k] = 0.0;
  int ngrid = 0;
  bool validrad = false;
  float e8[8], s8[NS][8], en[8], sn[NS][8];
  float srcext1[NS], ext1 = 0.f;
  int last[NST == 0 ? 8 : 1];
  for (int c = 0; c < (NST == 0 ? 8 : 1); c++) last[c] = -1;
  RayCell c, n;
  auto gather = [&](const RayCell& b, float* e, float (*s)[8]) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      e[k] = a.ext[b.gp[k]];
      for (int m = 0; m < NST; m++) s[m][k] = dsrc[(size_t)b.gp[k] * LD + m * a.cst];
    }
  };
  first_ray_cell<REG>(a, start, c);
  gather(c, e8, s8);
  while (!validrad && c.cell >= 0) {
    ngrid++;
    if constexpr (NST == 0) {
      for (int k = 0; k < 8; k++) {
        bool fresh = true;
        for (int o = 0; o < 8; o++) fresh = fresh && last[o] != c.gp[k];
        if (fresh) {
          if (listed < pl->cap) pl->list[(size_t)ir * pl->cap + listed] = c.gp[k];
          listed++;
        }
      }
      for (int k = 0; k < 8; k++) last[k] = c.gp[k];
    }
    const double delx = (double)(c.hi[0] - c.lo[0]);
    const double dely = (double)(c.hi[1] - c.lo[1]);
    const double delz = (double)(c.hi[2] - c.lo[2]);
    const bool ipinx = (c.fl & 1) && !(a.open_x && ((cx > 0 && xe < xm) || (cx < 0 && xe > xm)));
    const bool ipiny = (c.fl & 2) && !(a.open_y && ((cy > 0 && ye < ym) || (cy < 0 && ye > ym)));
    const double sox = ipinx ? 1.0e20 : ((double)(bitx ? c.lo[0] : c.hi[0]) - xe) * cxinv;
    const double soy = ipiny ? 1.0e20 : ((double)(bity ? c.lo[1] : c.hi[1]) - ye) * cyinv;
    const double soz = ((double)(bitz ? c.lo[2] : c.hi[2]) - ze) * czinv;
    double so = fmin(sox, fmin(soy, soz));
    if (so < -eps) {
      if constexpr (NST > 0) atomicOr(a.errflag, 1);
      break;
    }
    int iface, jface;
    bool openbcface;
    if (sox <= soz && sox <= soy) {
      iface = 1 - bitx;
      jface = 1;
      openbcface = (c.fl & 1) && a.open_x;
    } else if (soy <= soz) {
      iface = 3 - bity;
      jface = 2;
      openbcface = (c.fl & 2) && a.open_y;
    } else {
      iface = 5 - bitz;
      jface = 3;
      openbcface = false;
    }
    if constexpr (REG) {
      // the next cell's values load while this one is integrated
      next_ray_cell(a, c, jface, bitx, bity, bitz, n);
      if (n.cell >= 0) {
        load_ray_cell<true>(a, n);
        gather(n, en, sn);
      }
    }
    const double invdelx = delx <= 0.0 ? 1.0 : 1.0 / delx;
    const double invdely = dely <= 0.0 ? 1.0 : 1.0 / dely;
    const double invdelz = 1.0 / delz;
    const double px1 = c.lo[0], py1 = c.lo[1], pz1 = c.lo[2];
    double u = (xe - px1) * invdelx, v = (ye - py1) * invdely, w = (ze - pz1) * invdelz;
    // the entry values: interpolated in this cell (CORRECTINTERPOLATE, and
    // always in the first), else those the ray left the last cell with
    if (a.correct_interp || ngrid == 1) {
      for (int k = 0; k < NST; k++) srcext1[k] = trilin(s8[k], u, v, w);
      if constexpr (NST > 0) srcext1[0] = fmaxf(0.0f, srcext1[0]);
      ext1 = trilin(e8, u, v, w);
    }
    double xn = xe + so * cx, yn = ye + so * cy, zn = ze + so * cz;
    u = (xn - px1) * invdelx;
    v = (yn - py1) * invdely;
    w = (zn - pz1) * invdelz;
    const float extn = trilin(e8, u, v, w);
    const double taugrid = so * 0.5 * (double)(ext1 + extn);
    const int ntau = max(1, 1 + (int)(taugrid / a.tautol));
    const double dels = so / ntau;
    for (int it = 1; it <= ntau; it++) {
      const double s = it * dels;
      u = (xe + s * cx - px1) * invdelx;
      v = (ye + s * cy - py1) * invdely;
      w = (ze + s * cz - pz1) * invdelz;
      const float ext0 = trilin(e8, u, v, w);
      float srcext0[NS];
      for (int k = 0; k < NST; k++) srcext0[k] = trilin(s8[k], u, v, w);
      if constexpr (NST > 0) srcext0[0] = fmaxf(0.0f, srcext0[0]);
      const double ext = (double)(0.5f * (ext0 + ext1));
      double absc, trc;
      if (ext != 0.0) {
        const double tau = ext * dels;
        absc = tau * (1.0 - 0.5 * tau * (1.0 - (double)0.33333333333f * tau));
        trc = 1.0 - absc;
        for (int k = 0; k < NST; k++) {
          const double src = ((double)(0.5f * (srcext0[k] + srcext1[k])) +
                              (double)(0.08333333333f * (ext0 * srcext1[k] - ext1 * srcext0[k])) * dels *
                                  (1.0 - (double)(0.05f * (ext1 - ext0)) * dels)) / ext;
          radiance[k] = radiance[k] + transmit * src * absc;
        }
      } else {
        absc = 0.0;
        trc = 1.0;
      }
      transmit = transmit * trc;
      ext1 = ext0;
      for (int k = 0; k < NST; k++) srcext1[k] = srcext0[k];
    }
    int kface = iface, ic = c.cell;
    bool zface = iface >= 4;
    if constexpr (!REG) {
      // a face onto smaller cells continues down the neighbour's tree, and the
      // boundary interpolation takes that smaller face (NEXT_CELL)
      const int nbv = a.g.neighptr[(size_t)c.cell * 6 + iface];
      n.cell = nb_smaller(nbv) ? next_cell_down(a.g, nb_cell(nbv), iface, jface, xn, yn, zn) : nbv;
      if (n.cell >= 0) load_ray_cell<false>(a, n);
      if (openbcface || nb_smaller(nbv)) {
        kface = iface ^ 1;
        ic = n.cell;
        zface = false;
      }
    } else {
      zface = zface && !openbcface;
    }
    if (n.cell >= 0) {
      if (jface == 1) xn = bitx ? n.hi[0] : n.lo[0];
      else if (jface == 2) yn = bity ? n.hi[1] : n.lo[1];
      else zn = bitz ? n.hi[2] : n.lo[2];
    }
    if (transmit < a.transcut || ngrid > maxcross) {
      validrad = true;
    } else if (n.cell < 0 && zface) {
      validrad = true;
      if constexpr (NST == 0) break;
      // FIND_BOUNDARY_RADIANCE (shdomsub2.f:2748-2863), Lambertian surface
      const int8_t tab[6][4] = {{0, 2, 4, 6}, {1, 3, 5, 7}, {0, 1, 4, 5},
                                {2, 3, 6, 7}, {0, 1, 2, 3}, {4, 5, 6, 7}};
      float X[4], Y[4], R[4];
      for (int j = 0; j < 4; j++) {
        const int ip = a.g.gridptr[(size_t)ic * 8 + tab[kface][j]];
        X[j] = P[ip * 3];
        Y[j] = P[ip * 3 + 1];
        if ((float)mu2 < 0.0f) {
          R[j] = topv;
        } else {
          const int b = a.bot_index[ip];
          if (b < 0) atomicOr(a.errflag, 2);
          R[j] = b < 0 ? 0.0f : a.bcrad_bot[b];
        }
      }
      const float ub = (X[1] - X[0] > 0.0f) ? (float)((xn - X[0]) / (double)(X[1] - X[0])) : 0.0f;
      const float vb = (Y[2] - Y[0] > 0.0f) ? (float)((yn - Y[0]) / (double)(Y[2] - Y[0])) : 0.0f;
      const float radbnd = (1 - ub) * (1 - vb) * R[0] + ub * (1 - vb) * R[1] +
                           (1 - ub) * vb * R[2] + ub * vb * R[3];
      if (!a.nosurface) radiance[0] = radiance[0] + transmit * (double)radbnd;
    } else {
      if constexpr (!REG)
        if (n.cell >= 0) gather(n, en, sn);
      c = n;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        e8[k] = en[k];
        for (int m = 0; m < NST; m++) s8[m][k] = sn[m][k];
      }
    }
    xe = xn;
    ye = yn;
    ze = zn;
  }
  for (int k = 0; k < NST; k++) a.out[(size_t)ir * NST + k] = (float)radiance[k];
  if constexpr (NST == 0) {
    pl->cnt[ir] = min(listed, pl->cap);
    if (listed > pl->cap) atomicOr(pl->over, 1);
  }
}

template <int NST, bool REG>
__global__ __launch_bounds__(64) void k_render(RayArgs a) {
  const int ir = blockIdx.x * blockDim.x + threadIdx.x;
  if (ir < a.nrays) render_ray<NST, REG>(a, nullptr, ir);
}

template <bool REG>
__global__ __launch_bounds__(64) void k_ray_pairs(RayArgs a, PairArgs p) {
  const int ir = blockIdx.x * blockDim.x + threadIdx.x;
  if (ir < a.nrays) render_ray<0, REG>(a, &p, ir);
}

// The direction source of the listed pairs, as k_sh_to_do and the finish
// kernels give it for every point: 16 lanes a pair, the ray's harmonics in
// registers, a source row read as float4 (64 terms a step, up to NS).  With a
// direction per ray the full table takes npts x nrays products and several
// passes over npts x nrays words (61 x 61 rays of 64 x 64 x 40 points: 3.45 ms of
// GEMM and 10.5 ms of finish), a ray meets a few hundred points.  Rows are laid
// out by direction, so the points along a ray lie close together.
constexpr int PAIR_SEGS = 4;   // blocks per ray
constexpr int PAIR_LANES = 16;
template <bool GRAD>
__global__ __launch_bounds__(64) void k_pair_source(RayArgs a, PairArgs p) {
  const int ray = blockIdx.x, seg = blockIdx.y;
  const int n = p.cnt[ray], d = a.dir_of_ray[ray];
  const int lane = threadIdx.x & (PAIR_LANES - 1), g = threadIdx.x / PAIR_LANES;
  float4 y[8];
  const float* yr = p.Yd + (size_t)d * p.ld + 4 * lane;
#pragma unroll
  for (int i = 0; i < 8; i++)
    y[i] = 64 * i < p.ld ? *reinterpret_cast<const float4*>(yr + 64 * i) : make_float4(0.f, 0.f, 0.f, 0.f);
  const float g0 = lane <= p.ml ? p.G[(size_t)d * (p.ml + 1) + lane] : 0.f;
  for (int k = seg * 4 + g; k < n; k += 4 * PAIR_SEGS) {
    const int q = p.list[(size_t)ray * p.cap + k];
    const int ns = p.ns[q];
    float v = 0.f, ss = 0.f;
    if (!p.single_scatter) {
      const float* sr = p.S + (size_t)q * p.ld + 4 * lane;
#pragma unroll
      for (int i = 0; i < 8; i++)
        if (64 * i < ns) {
          const float4 s = *reinterpret_cast<const float4*>(sr + 64 * i);
          v = fmaf(s.x, y[i].x, fmaf(s.y, y[i].y, fmaf(s.z, y[i].z, fmaf(s.w, y[i].w, v))));
        }
      if (p.tms_on && ns > 0) {
        const int ls = p.lofj[ns - 1];
        const float* t = p.tms + (size_t)q * (p.ml + 1);
        if (lane <= ls) v = fmaf(-t[lane], g0, v);
        for (int l = lane + PAIR_LANES; l <= ls; l += PAIR_LANES)
          v = fmaf(-t[l], p.G[(size_t)d * (p.ml + 1) + l], v);
      }
    }
    if (p.tms_on)
      for (int t = p.ss_off[q] + lane; t < p.ss_off[q + 1]; t += PAIR_LANES)
        ss = fmaf(p.ss_coef[t], p.ssd[(size_t)d * p.numphase + p.ss_iph[t]], ss);
    v += ss;
#pragma unroll
    for (int m = PAIR_LANES / 2; m > 0; m >>= 1) {
      v += __shfl_xor(v, m);
      if (GRAD) ss += __shfl_xor(ss, m);
    }
    if (lane == 0) {
      const size_t o = q * a.ps + d * a.ds;
      const float e = a.ext[q];
      p.dsrc[o] = v * e;
      if (GRAD) {
        p.srcpre[o] = v;
        p.ss8[o] = ss * e;
        p.bsrc[o] = 0.0;
      }
    }
  }
}

// Spherical harmonics of one direction (YLMALL_UNPOL, shdomsub2.f:4490-4539; the
// Wigner functions d^l_{m0} by their three-term recurrence in FP64, one m per
// lane), the truncated single-scatter factors and the phase table at the
// scattering angle, one wavefront per direction: 1.8 us each on a host core
// before (7.8 ms for 4394 directions).
__global__ __launch_bounds__(64) void k_direction_tables(DirectionArgs a) {
#pragma clang fp contract(off)
  __shared__ float yl[512];
  const int d = blockIdx.x, lane = threadIdx.x;
  float* row = a.Yd + (size_t)d * a.ld;
  if (d >= a.nd) {
    for (int j = lane; j < a.ld; j += 64) row[j] = 0.f;
    return;
  }
  const double PI = acos(-1.0);
  const double mu2 = a.dirs[2 * d], phi2 = a.dirs[2 * d + 1];
  const double x = (double)(float)mu2, fct = 1.0 / sqrt(2.0 * PI);
  auto index = [&](int l, int m) { return l <= a.mm ? l * (l + 1) + m : (2 * a.mm + 1) * l - a.mm * a.mm + m; };
  for (int m = lane; m <= a.mm; m += 64) {
    double cosm = 1.0, sinm = 0.0, cur = 1.0, old = 0.0;
    if (m > 0) {
      // (single-precision angle and values, as the reference's COS and SIN)
      const float ang = (float)m * (float)phi2;
      cosm = (double)(float)cos((double)ang);
      sinm = (double)(float)sin((double)ang);
      double prod = 1.0;
      for (int k = 1; k <= m; k++) prod *= sqrt((m + k) / (double)k);
      cur = (m % 2 ? -1.0 : 1.0) * prod * pow(0.5 * sqrt((1.0 - x) * (1.0 + x)), (double)m);
    }
    for (int l = m; l <= a.ml; l++) {
      const double v = fct * (sqrt(l + 0.5) * cur);
      yl[index(l, m)] = (float)((cosm - sinm) * v);
      yl[index(l, -m)] = (float)((cosm + sinm) * v);
      double nxt;
      if (m == 0)
        nxt = l == 0 ? x : ((2 * l + 1) * x * cur - l * old) / (l + 1);
      else
        nxt = ((2 * l + 1) * x * cur - sqrt((double)(l * l - m * m)) * old) /
              sqrt((double)((l + 1) * (l + 1) - m * m));
      old = cur;
      cur = nxt;
    }
  }
  __syncthreads();
  for (int j = lane; j < a.ld; j += 64) row[j] = j < a.nlm ? yl[j] : 0.f;
  for (int l = lane; l <= a.ml; l += 64) {
    double g = 0.0;
    for (int j = l == 0 ? 0 : nterms_l(l - 1, a.mm); j < nterms_l(l, a.mm); j++)
      g += (double)yl[j] * (double)a.ysun[j];
    a.G[(size_t)d * (a.ml + 1) + l] = (float)g;
  }
  if (!a.phasetab) {
    for (int k = lane; k < a.numphase; k += 64) a.ssd[(size_t)d * a.numphase + k] = 0.f;
    return;
  }
  double cosscat = (double)a.solarmu * mu2 + sqrt((double)(1.0f - a.solarmu * a.solarmu) * (1.0 - mu2 * mu2)) *
                                                 cos((double)a.solaraz - phi2);
  cosscat = fmax(fmin(1.0, cosscat), -1.0);
  float f = (float)((a.nsa - 1) * (acos(cosscat) / PI) + 1);
  const int j = min(a.nsa - 1, (int)f);
  f = f - (float)j;
  for (int k = lane; k < a.numphase; k += 64) {
    const float* t = a.phasetab + (size_t)k * a.nsa + j;
    a.ssd[(size_t)d * a.numphase + k] = (1 - f) * t[-1] + f * t[0];
  }
  for (int k = lane; k < a.dnumphase; k += 64) {
    const float* t = a.dphasetab + (size_t)k * a.nsa + j;
    a.dssd[(size_t)d * a.dnumphase + k] = (1 - f) * t[-1] + f * t[0];
  }
}

// Surface radiance from the final fluxes (RENDER :201-209).
__global__ void k_render_bottom(const float* __restrict__ fluxes, const float* __restrict__ dirflux,
                                const int32_t* __restrict__ bcbot, int nbot, float albpi,
                                float* __restrict__ bcrad) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbot) return;
  const int p = bcbot[b];
  bcrad[b] = albpi * (dirflux[p] + fluxes[p]);
}

void launch_dir_source_finish(hipStream_t st, const float* raw, int ldd, int ndir, const float* ext,
                              const int* ns, const int* lofj, const float* tms, const float* G,
                              const int32_t* ss_off, const int32_t* ss_iph, const float* ss_coef,
                              const float* ssd, int numphase, int ml, int npts, int single_scatter,
                              int tms_on, float* dsrc) {
  const int n = npts * ndir;
  k_dir_source_finish<<<(n + 255) / 256, 256, 0, st>>>(raw, ldd, ndir, ext, ns, lofj, tms, G, ss_off,
                                                        ss_iph, ss_coef, ssd, numphase, ml, npts,
                                                        single_scatter, tms_on, dsrc);
}

void launch_render(hipStream_t st, const RayArgs& a) {
  const int nb = (a.nrays + 63) / 64;
  const bool reg = a.g.treeptr == nullptr;
  if (a.nst == 3)
    reg ? k_render<3, true><<<nb, 64, 0, st>>>(a) : k_render<3, false><<<nb, 64, 0, st>>>(a);
  else
    reg ? k_render<1, true><<<nb, 64, 0, st>>>(a) : k_render<1, false><<<nb, 64, 0, st>>>(a);
}

void launch_ray_pairs(hipStream_t st, const RayArgs& a, const PairArgs& p) {
  const int nb = (a.nrays + 63) / 64;
  a.g.treeptr == nullptr ? k_ray_pairs<true><<<nb, 64, 0, st>>>(a, p) : k_ray_pairs<false><<<nb, 64, 0, st>>>(a, p);
}

void launch_pair_source(hipStream_t st, const RayArgs& a, const PairArgs& p) {
  const dim3 grid(a.nrays, PAIR_SEGS);
  if (p.srcpre)
    k_pair_source<true><<<grid, 64, 0, st>>>(a, p);
  else
    k_pair_source<false><<<grid, 64, 0, st>>>(a, p);
}

void launch_direction_tables(hipStream_t st, const DirectionArgs& a) {
  k_direction_tables<<<a.ldd, 64, 0, st>>>(a);
}

void launch_dir_source_finish_pol(hipStream_t st, const float* raw, int ldd, int cst, int ndir, const float* ext,
                                  const int* ns, const int* lofj, const float* tms, const float* tms5,
                                  const float* G3, const int32_t* ss_off, const int32_t* ss_iph,
                                  const float* ss_coef, const float* ssd, const float* ssq, const float* ssu,
                                  int numphase, int ml, int npts, int single_scatter, int tms_on, float* dsrc) {
  const int n = npts * ndir;
  k_dir_source_finish_pol<<<(n + 255) / 256, 256, 0, st>>>(raw, ldd, cst, ndir, ext, ns, lofj, tms, tms5, G3,
                                                            ss_off, ss_iph, ss_coef, ssd, ssq, ssu, numphase,
                                                            ml, npts, single_scatter, tms_on, dsrc);
}

void launch_render_bottom(hipStream_t st, const float* fluxes, const float* dirflux,
                          const int32_t* bcbot, int nbot, float albpi, float* bcrad) {
  if (nbot <= 0) return;
  k_render_bottom<<<(nbot + 255) / 256, 256, 0, st>>>(fluxes, dirflux, bcbot, nbot, albpi, bcrad);
}

}  // namespace at3d
