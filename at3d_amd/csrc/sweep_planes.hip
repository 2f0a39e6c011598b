// Plane-ordered sweep of open base grids (BACK_INT_GRID3D_UNPOL,
// shdomsub1.f:3695-4032).
//
// On a tensor-product grid every point of an ordinate's interior steps to the
// same face of its upwind cell: the horizontal one (z), or the side facing x or
// y, whichever spacing over direction cosine is the shortest.  So a whole grid
// plane across that axis depends on the plane before it alone, and an ordinate
// takes as many dependent levels as the grid has planes (40 to 64 at 64 x 64 x
// 40, against 163 levels of the octants' common order), with every upwind value
// at a fixed offset: nothing about a step has to be recorded or read.  Points on
// the sides of the open domain keep to their side (independent-pixel columns):
// the step is the same with the neighbour off the side replaced by the point
// itself, and the first and last planes of an x or y ordinate are
// two-dimensional sweeps of their own.
//
// One workgroup per ordinate and Stokes component.  LDS holds the last plane's
// radiance, extinction and source and this plane's source (16 bytes a point);
// a thread owns the same points of every plane, so their offsets, edges and
// weights stay in registers.  The source rows come in the order SH->DO writes
// them: plane by plane, within a plane grouped by source class (its tiles of 64
// then stop their K loop early), scattered to their place through a 16-bit
// index that all ordinates of the axis share.  The next plane's loads fly while
// one is integrated.  Radiances go to the point-ordered row: whole planes for an
// x ordinate, runs of nz for y, and four planes at a time (16 bytes a point) for
// z.
//
// No one unit bounds it: at 64 x 64 x 40 the vector units issue 80 instructions a
// point (the transmission and source weights of cell_coefs and the interpolation,
// and the moves of scalars spilled to vector lanes) half of the time, the LDS is in use
// for 53 % of it, two thirds of that in bank conflicts of the 16-byte points, and a
// wavefront waits half of its life, mostly at the two barriers a plane.  Per
// hemisphere, against k_sweep_ring: 64 x 64 x 40, 177 ordinates 138 against 253 us;
// 32 x 32 x 32, 45 ordinates 37 against 92;
// 48 x 48 x 32, cold 84 against 156 and no records pass (730 us a solve).  Plane order
// also feeds SH->DO longer runs of one class: 128 against 153 us at 64 x 64 x 40.
//
// Planes past PLANE_POINTS_MAX go in strips of rows, one after the other in the
// ordinate's direction, each through all planes: a strip reads of the one before
// only its last row, whose radiances and sources stay in LDS (8 bytes a line and
// plane).  More points a thread instead spill registers (96 x 96 planes, ten a
// thread: 1012 us a hemisphere; 128 x 128, 16: 16.8 ms).  Against the ring:
// 96 x 96 x 48, 177 ordinates, 405 us for 984; 128 x 128 x 64 with three Stokes
// components 2.0 ms for 5.77.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "cell_coefs.h"
#include "kernels.h"

namespace at3d {

struct __attribute__((packed, aligned(4))) Vec4 {
  float x, y, z, w;
};

// Element i of a row by a 32-bit byte offset from a uniform base (one register
// an address; rows are under 2^30 elements).
template <typename V, typename U>
__device__ __forceinline__ V& at(U* row, uint32_t i) {
  using B = std::conditional_t<std::is_const_v<U>, const char, char>;
  return *reinterpret_cast<V*>(reinterpret_cast<B*>(row) + i * (uint32_t)sizeof(U));
}

// A point in LDS: {radiance, extinction} of its plane, source of the even and of
// the odd planes.
struct PlanePoint {
  float2 re;
  float s[2];
};
// K points a thread. ZT: an ordinate that goes by z.  STRIPS: planes of more than
// one strip.
template <int T, int K, bool ZT, bool STRIPS>
__device__ __forceinline__ void sweep_planes(const SweepArgs& a, const PlaneArgs& p, int col, int kst, float4* lds) {
  const OrdGeom og = a.ordg[col];
  const int code = p.col_type[col], t = code & 3;
  const int nx = a.nx1, ny = a.ny1, nz = a.nz;
  const int na = ZT ? ny : nz, nb = ZT ? nx : (t == 1 ? ny : nx), N = ZT ? nz : (t == 1 ? nx : ny);
  const int sb = STRIPS ? p.sb[t] : nb;   // rows (of na points) a strip
  const int lbit = ZT ? og.bitz : (t == 1 ? og.bitx : og.bity);
  const int abit = ZT ? og.bity : og.bitz, bbit = ZT ? og.bitx : (t == 1 ? og.bity : og.bitx);
  // upwind neighbours: a + ua, b + ub
  const int k0 = lbit ? 0 : N - 1, kstep = lbit ? 1 : -1;
  const int ua = abit ? -1 : 1, ub = bbit ? -1 : 1, uba = ub * na;
  const int zstart = og.bitz ? 0 : nz - 1, uz = og.bitz ? -1 : 1;
  const int up = og.bitz;
  const int tid = threadIdx.x;
  float4* tab = lds;   // per z level
  // the strip's points, and on the side upwind the last strip's row next to it
  // (of the same planes): radiance and source kept in H, [N][na]
  PlanePoint* P = reinterpret_cast<PlanePoint*>(lds + nz) + (STRIPS && bbit ? na : 0);
  float2* H = reinterpret_cast<float2*>(lds + nz + (sb + 1) * na);
  // the surface radiances along the plane's z boundary (x and y ordinates)
  float* B = STRIPS ? reinterpret_cast<float*>(H + (sb < nb ? N * na : 0)) : reinterpret_cast<float*>(lds + nz + sb * na);
  const double cx = fabs(og.cx), cy = fabs(og.cy), cz = fabs(og.cz);
  const double hx = p.dx * fabs(og.cxinv), hy = p.dy * fabs(og.cyinv);
  for (int z = tid; z < nz; z += T) {
    const double dz = z == zstart ? 1.0 : fabs((double)a.zgrid[z + uz] - (double)a.zgrid[z]), hz = dz * fabs(og.czinv);
    // .x path, .y and .z weights of a's and b's neighbours; .w on a side, the
    // weight of the neighbour in its own plane
    const double hb = t == 1 ? hy : hx, cb = t == 1 ? cy / p.dy : cx / p.dx;
    tab[z] = ZT       ? make_float4((float)hz, (float)(hz * cy / p.dy), (float)(hz * cx / p.dx), 0.f)
             : t == 1 ? make_float4((float)hx, (float)(hx * cz / dz), (float)(hx * cy / p.dy), 0.f)
                      : make_float4((float)hy, (float)(hy * cz / dz), (float)(hy * cx / p.dx), 0.f);
    if (!ZT) tab[z].w = (float)((code & 4) ? hb * cz / dz : hz * cb);
  }
  const float* se = a.srcext + kst * a.pdo + (size_t)col * a.ldp;
  float* rad = a.rad + kst * a.pdo + (size_t)col * a.ldp;
  const uint16_t* pidx = p.pidx + (size_t)t * a.npts;
  const float* ext = p.ext + (size_t)t * a.npts;
  const float sky = kst ? 0.0f : a.skyrad[col];
  // the surface radiance below (x, y); boundary points are in point order
  auto bottom = [&](int x, int y) { return kst ? 0.0f : a.bcrad_bot[y + ny * x]; };
  auto boundary = [&](int kc, int b) { return !up ? sky : t == 1 ? bottom(kc, b) : bottom(b, kc); };
  // this thread's points: s = tid + k T (the last one again past the end)
  const int stride = ZT ? 1 : (t == 1 ? ny * nz : nz);   // of the point index from plane to plane
  // Radiances go out behind the next barrier where a thread stores three or more
  // single words a plane: 64 x 64 x 40, 138 us a hemisphere for 154, 96 x 96 x 48
  // 405 for 451; fewer, or a z ordinate's four planes at a time, the other way
  // (32^3 41 for 37 us, 96 x 96 x 48 468).
  constexpr bool LATE = !ZT && K >= 3;
  constexpr int KB = (K + 1) / 2;   // surface radiances a thread: a row has two points at least
  const int nstrips = STRIPS ? (nb + sb - 1) / sb : 1;
  __syncthreads();
  for (int strip = 0; strip < nstrips; strip++) {
    const int b0 = STRIPS ? (bbit ? strip : nstrips - 1 - strip) * sb : 0, rows = STRIPS ? min(sb, nb - b0) : nb;
    const int M = na * rows, g0 = na * b0;
    uint32_t ea = 0, eb = 0;   // on a side across a (x and y ordinates: on the z boundary), across b
    uint32_t el_row = 0;       // in the row that the next strip reads (the last downwind)
    int goff[ZT ? 1 : K];
    float wa[ZT ? 1 : K];
    // the neighbours' offsets in points: a's in the low half, b's in the high one
    int nbr[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
      if (k * T >= M) break;
      const int s = min(tid + k * T, M - 1), bl = s / na, ai = s - bl * na, bi = b0 + bl;
      ea |= (uint32_t)(ZT ? ai == 0 || ai == na - 1 : ai == zstart) << k;
      eb |= (uint32_t)(bi == 0 || bi == nb - 1) << k;
      if constexpr (STRIPS) el_row |= (uint32_t)(tid + k * T < M && bl == (bbit ? rows - 1 : 0)) << k;
      nbr[k] = (ZT && (ai == 0 || ai == na - 1) ? 0 : ua & 0xffff) | ((bi == 0 || bi == nb - 1 ? 0 : uba) * 65536);
      if constexpr (!ZT) {
        goff[k] = t == 1 ? g0 + s : ai + nz * ny * bi;
        wa[k] = ai == zstart ? 0.f : tab[ai].y;
        if (ai == zstart) nbr[k] = (nbr[k] & ~0xffff) | bl;   // (a boundary value replaces the sum: its place in B)
      }
    }
    float sl[K], el[K], ec[K], val[K], bl[ZT ? 1 : KB];
    uint16_t il[K];
    auto load = [&](int kc) {
      // (sources strip by strip, extinctions whole planes)
      const int base = g0 * N + kc * M, ebase = kc * na * nb + g0;
#pragma unroll
      for (int k = 0; k < K; k++) {
        if (k * T >= M) break;
        const int s = min(tid + k * T, M - 1);
        sl[k] = at<const float>(se, base + s);
        il[k] = at<const uint16_t>(pidx, base + s);
        el[k] = at<const float>(ext, ebase + s);
      }
      if constexpr (!ZT)   // the surface radiances of the plane's z boundary
        if (up) {
#pragma unroll
          for (int k = 0; k < KB; k++)
            if (tid + k * T < rows) bl[k] = boundary(kc, b0 + tid + k * T);
        }
    };
    // The row of the strip before: each line of it is fetched by the thread that
    // owns the same line of this strip's last row (eh: its extinction), so that
    // H's entry is read and then written by one thread.
    const bool halo = STRIPS && strip > 0, last = !STRIPS || strip + 1 == nstrips;
    const int own_row = (bbit ? rows - 1 : 0) * na, halo_row = bbit ? -na : M;
    float eh = 0.f;
    auto load_halo = [&](int kc) {
      if (!halo || el_row == 0) return;
#pragma unroll
      for (int k = 0; k < K; k++)
        if ((el_row >> k) & 1)
          eh = at<const float>(ext, kc * na * nb + g0 + halo_row + tid + k * T - own_row);
    };
    float h1[ZT ? K : 1], h2[ZT ? K : 1], h3[ZT ? K : 1];   // the last three planes' radiances
    int held = 0;
    // plane l's radiances (val) out to the point-ordered row
    auto put = [&](int kc, int l) {
      if constexpr (ZT) {
        held++;
        const bool flush = l == N - 1 || (kc & 3) == (kstep < 0 ? 0 : 3);
        auto each = [&](auto&& f) {
#pragma unroll
          for (int k = 0; k < K; k++) {
            if (k * T >= M) break;
            f(k, (uint32_t)(nz * (g0 + min(tid + k * T, M - 1)) + kc));
          }
        };
        if (flush && held == 4) {
          each([&](int k, uint32_t o) {
            Vec4 v;
            v.x = kstep < 0 ? val[k] : h3[k];
            v.y = kstep < 0 ? h1[k] : h2[k];
            v.z = kstep < 0 ? h2[k] : h1[k];
            v.w = kstep < 0 ? h3[k] : val[k];
            at<Vec4>(rad, kstep < 0 ? o : o - 3) = v;
          });
        } else if (flush) {
          each([&](int k, uint32_t o) {
            at<float>(rad, o) = val[k];
            if (held > 1) at<float>(rad, o - kstep) = h1[k];
            if (held > 2) at<float>(rad, o - 2 * kstep) = h2[k];
          });
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
          h3[k] = h2[k];
          h2[k] = h1[k];
          h1[k] = val[k];
        }
        if (flush) held = 0;
      } else {
#pragma unroll
        for (int k = 0; k < K; k++) {
          if (k * T >= M) break;
          at<float>(rad, (uint32_t)(goff[k] + kc * stride)) = val[k];
        }
      }
    };
    load(k0);
    if (STRIPS && !ZT) load_halo(k0);
    for (int L = 0; L < N + (LATE || (STRIPS && !ZT)); L++) {   // (past the last plane: its radiances, its row)
      const int kc = k0 + L * kstep, par = L & 1;
      const bool side = !ZT && (L == 0 || L == N - 1);
      if (L < N) {
        // the last plane's radiance and extinction (a side's own extinction), this
        // plane's source
#pragma unroll
        for (int k = 0; k < K; k++) {
          if (k * T >= M) break;
          const int s = min(tid + k * T, M - 1);
          if (L > 0 && !side) P[s].re = make_float2(val[k], ec[k]);
          P[il[k]].s[par] = sl[k];
          ec[k] = el[k];
          if constexpr (!ZT)
            if (side) P[s].re.y = ec[k];
        }
        if constexpr (!ZT)
          if (up) {
#pragma unroll
            for (int k = 0; k < KB; k++)
              if (tid + k * T < rows) B[tid + k * T] = bl[k];
          }
        if constexpr (STRIPS) {
          // the plane before (a side's: this plane) of the last strip's row, and this
          // strip's own for the next one
          if (el_row && (L > 0 || side)) {
#pragma unroll
            for (int k = 0; k < K; k++) {
              if (!((el_row >> k) & 1)) continue;
              const int s = tid + k * T, ai = s - own_row;
              if (halo) {
                const float2 h = H[(side ? kc : kc - kstep) * na + ai];
                P[halo_row + ai].re = make_float2(h.x, eh);
                P[halo_row + ai].s[side ? par : par ^ 1] = h.y;
              }
              if (!last && L > 0) H[(kc - kstep) * na + ai] = make_float2(val[k], P[s].s[par ^ 1]);
            }
          }
        }
      } else if constexpr (STRIPS && !ZT) {
        // the last side's row (before the barrier: the next strip writes P after it)
        if (el_row && !last) {
#pragma unroll
          for (int k = 0; k < K; k++)
            if ((el_row >> k) & 1)
              H[(kc - kstep) * na + tid + k * T - own_row] = make_float2(val[k], P[tid + k * T].s[par ^ 1]);
        }
      }
      lds_barrier();
      // (LATE: the last plane's radiances, then the next plane's loads; waiting for
      // the loads waits for stores between, which so have this plane's arithmetic
      // to complete)
      if constexpr (LATE)
        if (L > 0) put(kc - kstep, L - 1);
      if (L == N) break;
      if (L + 1 < N) {
        load(kc + kstep);
        if constexpr (STRIPS) load_halo(!ZT && L + 2 == N ? kc + kstep : kc);
      }
      if (ZT && L == 0) {
#pragma unroll
        for (int k = 0; k < K; k++) {
          if (k * T >= M) break;
          val[k] = up ? (kst ? 0.0f : a.bcrad_bot[g0 + min(tid + k * T, M - 1)]) : sky;   // y + ny x, as they are
        }
      } else if (!ZT && side) {
        if constexpr (!ZT) {
        // a side of the open domain: a two-dimensional sweep in z and the other
        // axis b.  Every point's source integral (in place of its radiance) and
        // transmission (of the source no longer needed) first, then the first
        // wavefront adds the transmitted radiances line by line: a line costs an
        // LDS round trip and three operations.
        const bool byb = (code & 4) != 0;
        const float hb = (float)(t == 1 ? hy : hx);
#pragma unroll
        for (int k = 0; k < K; k++) {
          if (k * T >= M) break;
          const int s = min(tid + k * T, M - 1), z = s - s / na * na;
          const bool edge = (eb >> k) & 1, preset = (ea >> k) & 1;
        const float bv = up && preset ? B[nbr[k] & 0xffff] : sky;
          // the corner upwind and its neighbour, weight w
          const bool viab = byb && !edge;
          const int su = preset ? s : viab ? s + uba : s + uz, du = preset || edge ? 0 : viab ? uz : uba;
          const float w = edge ? 0.f : tab[z].w;
          const float so = viab ? hb : (float)(fabs((double)a.zgrid[preset ? z : z + uz] - (double)a.zgrid[z]) * fabs(og.czinv));
          const float ea0 = P[su].re.y, sa0 = P[su].s[par];
          const float e0 = fmaf(w, P[su + du].re.y - ea0, ea0);
          const float s0 = fmaf(w, P[su + du].s[par] - sa0, sa0);
          float b0, b1, trc;
          cell_coefs(e0, ec[k], so, b0, b1, trc);
          const float sv = b0 * s0 + b1 * P[s].s[par];
          P[s].re.x = preset ? bv : (kst ? sv : fmaxf(0.f, sv));
          P[s].s[par ^ 1] = preset ? 0.f : trc;
        }
        lds_barrier();
        if (tid < 64) {
          auto step = [&](int s, int su, int du, float w) {
            const float r0 = P[su].re.x, r1 = P[su + du].re.x;
            P[s].re.x = fmaf(P[s].s[par ^ 1], fmaf(w, r1 - r0, r0), P[s].re.x);
          };
          if (!byb) {
            for (int z = zstart - uz; z >= 0 && z < nz; z -= uz) {
              const float w = tab[z].w;
              for (int b = tid; b < rows; b += 64) {
                const bool edge = b0 + b == 0 || b0 + b == nb - 1;
                step(z + na * b, z + uz + na * b, edge ? 0 : uba, edge ? 0.f : w);
              }
              wave_lds_fence();
            }
          } else {
            const int be = (tid ? nb - 1 : 0) - b0;   // the open domain's own columns
            if (tid < 2 && be >= 0 && be < rows) {
              const int b = be;
              for (int z = zstart - uz; z >= 0 && z < nz; z -= uz) step(z + na * b, z + uz + na * b, 0, 0.f);
            }
            wave_lds_fence();
            for (int i = 0; i < rows; i++) {
              const int b = bbit ? i : rows - 1 - i;
              if (b0 + b == 0 || b0 + b == nb - 1) continue;
              for (int z = tid; z < nz; z += 64)
                if (z != zstart) step(z + na * b, z + na * (b + ub), uz, tab[z].w);
              wave_lds_fence();
            }
          }
        }
        lds_barrier();
#pragma unroll
        for (int k = 0; k < K; k++) {
          if (k * T >= M) break;
          val[k] = P[min(tid + k * T, M - 1)].re.x;
        }
        }
      } else {
        const float4 g = tab[ZT ? kc : 0];
        const float so = g.x, wz = g.y, wb = g.z;
#pragma unroll
        for (int k = 0; k < K; k++) {
          if (k * T >= M) break;
          const int s = min(tid + k * T, M - 1);
          const float w1 = ZT ? wz : wa[k];
          const float f3 = w1 * wb, f1 = w1 - f3, f2 = wb - f3, f0 = 1.f - w1 - f2;
          const bool preset = !ZT && ((ea >> k) & 1);
          const int oa = preset ? 0 : (int)(int16_t)nbr[k], ob = nbr[k] >> 16;
          const PlanePoint *q0 = P + s, *q1 = q0 + oa, *q2 = q0 + ob, *q3 = q1 + ob;
          const float2 v0 = q0->re, v1 = q1->re, v2 = q2->re, v3 = q3->re;
          const float c0 = q0->s[par ^ 1], c1 = q1->s[par ^ 1], c2 = q2->s[par ^ 1], c3 = q3->s[par ^ 1];
          const float e0 = f0 * v0.y + f1 * v1.y + f2 * v2.y + f3 * v3.y;
          const float s0 = f0 * c0 + f1 * c1 + f2 * c2 + f3 * c3;
          const float r0 = f0 * v0.x + f1 * v1.x + f2 * v2.x + f3 * v3.x;
          float b0, b1, trc;
          cell_coefs(e0, ec[k], so, b0, b1, trc);
          const float sv = b0 * s0 + b1 * q0->s[par];
          val[k] = (kst ? sv : fmaxf(0.f, sv)) + trc * r0;
          if (preset) val[k] = up ? B[nbr[k] & 0xffff] : sky;
        }
      }
      if constexpr (!LATE) put(kc, L);
      lds_barrier();
    }
  }
}

// KZ, KS: points a thread of planes across z, and across x or y.
template <int T, int KZ, int KS, bool STRIPS>
__global__ __launch_bounds__(T) void k_sweep_planes(SweepArgs a, PlaneArgs p, int col0) {
  if (a.stop && *a.stop) return;
  extern __shared__ float4 planes_lds[];
  const int col = col0 + blockIdx.x;
  if (blockIdx.y == 0 && col >= a.qu_only_from) return;
  if ((p.col_type[col] & 3) == 0)
    sweep_planes<T, KZ, true, STRIPS>(a, p, col, blockIdx.y, planes_lds);
  else
    sweep_planes<T, KS, false, STRIPS>(a, p, col, blockIdx.y, planes_lds);
}

// The extinction in each axis's plane order (plane by plane, within a plane by
// its natural index).
__global__ void k_plane_ext(const float* __restrict__ ext, float* __restrict__ out, int nx, int ny, int nz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y, n = nx * ny * nz;
  if (i >= n) return;
  int q;
  if (t == 0) {          // [z][x][y]
    const int z = i / (nx * ny), s = i - z * nx * ny;
    q = z + nz * s;
  } else if (t == 1) {   // [x][y][z]
    q = i;
  } else {               // [y][x][z]
    const int y = i / (nx * nz), s = i - y * nx * nz, x = s / nz;
    q = s - x * nz + nz * (y + ny * x);
  }
  out[(size_t)t * n + i] = ext[q];
}

void launch_plane_ext(hipStream_t st, const float* ext, float* out, int nx, int ny, int nz) {
  k_plane_ext<<<dim3((nx * ny * nz + 255) / 256, 3), 256, 0, st>>>(ext, out, nx, ny, nz);
}

// Threads and points per thread: 1024 threads where a plane fills them, fewer
// for small planes (fewer wavefronts at each barrier).
struct PlaneShape {
  const void* f;
  void (*go)(dim3, size_t, hipStream_t, const SweepArgs&, const PlaneArgs&, int);
};
template <int T, int KZ, int KS, bool STRIPS = false>
static PlaneShape plane_shape() {
  return {reinterpret_cast<const void*>(k_sweep_planes<T, KZ, KS, STRIPS>),
          [](dim3 g, size_t lds, hipStream_t st, const SweepArgs& a, const PlaneArgs& p, int c0) {
            k_sweep_planes<T, KZ, KS, STRIPS><<<g, T, lds, st>>>(a, p, c0);
          }};
}
static PlaneShape shape_of(int mz, int ms, bool strips) {
  if (strips) return plane_shape<1024, 3, 3, true>();
  const int m = mz > ms ? mz : ms;
  if (m <= 256) return plane_shape<256, 1, 1>();
  if (m <= 512) return plane_shape<512, 1, 1>();
  if (m <= 1024) return plane_shape<512, 2, 2>();
  if (mz <= 2048) {
    if (ms <= 2048) return plane_shape<1024, 2, 2>();
    return ms <= 3072 ? plane_shape<1024, 2, 3>() : plane_shape<1024, 2, 4>();
  }
  if (mz <= 3072) {
    if (ms <= 2048) return plane_shape<1024, 3, 2>();
    return ms <= 3072 ? plane_shape<1024, 3, 3>() : plane_shape<1024, 3, 4>();
  }
  if (ms <= 2048) return plane_shape<1024, 4, 2>();
  return ms <= 3072 ? plane_shape<1024, 4, 3>() : plane_shape<1024, 4, 4>();
}

int sweep_planes_max_lds(int mz, int ms, bool strips, size_t lds) {
  return hipFuncSetAttribute(shape_of(mz, ms, strips).f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess
             ? 0
             : 1;
}

void launch_sweep_planes(hipStream_t st, const SweepArgs& a, const PlaneArgs& p, int col0, int ncol, int mz, int ms,
                         bool strips, size_t lds) {
  if (ncol <= 0) return;
  shape_of(mz, ms, strips).go(dim3(ncol, a.nst), lds, st, a, p, col0);
}

}  // namespace at3d
