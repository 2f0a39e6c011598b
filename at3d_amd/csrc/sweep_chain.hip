// Point-ordered sweep of small grids from per-ordinate records
// (BACK_INT_GRID3D_UNPOL, shdomsub1.f:3695-4032).
//
// Periodic grids (whose multi-cell traces depend on the points swept just
// before) and grids refined by cell splitting keep the point order.  What a
// point's radiance takes from the sweep itself is linear: the four corners of
// the face its characteristic stops on, times fixed weights and the fixed
// transmission of the path; everything else of the trace depends on the source
// alone.  So a sweep is two launches: k_chain_source integrates the source
// along every characteristic of every ordinate at once (nothing waits), and
// k_sweep_chain adds the transmitted corner radiances, one wavefront per
// ordinate with the ordinate's radiances in LDS.
//
// The order of k_sweep_chain is by the dependency levels of its own ordinate.
// The levels the host planner gives a whole octant hold every ordinate's
// dependencies together: 4080 of them on the 16^3 periodic grid at NMU 8, where
// most ordinates alone have 15 to 325 and eight oblique ones 1554 to 3588.  A
// level costs one LDS round trip and five dependent FP64 operations (80 ns);
// k_sweep_columns, which traces at every level behind a workgroup barrier, takes
// 2.7 us.  Measured per hemisphere on that grid: 11.1 ms before, 0.33 ms now
// (0.29 of it k_sweep_chain); a 17 x 15 x 12 grid refined to about 8000 points
// 1.4 ms before, 0.12 now.  Weights, transmissions and sums are FP64 as in the
// general trace, the row is rounded to FP32 at every point; the transmission is
// multiplied into the weights and the sum is fused, which differs from the
// general trace by 1e-16 before that rounding.
#include <hip/hip_runtime.h>

#include "cell_coefs.h"
#include "kernels.h"

namespace at3d {

// The characteristic of one point back to the face whose corners are known
// (sweep_general without the radiances): per cell step `step(t, f)` sees the
// step and its face weights; returns the errflag bits of a bad trace.
template <typename Step>
__device__ inline int chain_walk(const SweepArgs& a, const OrdGeom& og, int o, int pt, int icell, TraceStep& t,
                                 Step&& step) {
  const int presetbit = og.bitz ? 2 : 1;
  const int32_t* rank = a.rank + (size_t)o * a.npts;
  const int rp = rank[pt];
  double xe = a.g.gridpos[pt * 3], ye = a.g.gridpos[pt * 3 + 1], ze = a.g.gridpos[pt * 3 + 2];
  for (int n = 0; n <= a.g.ncells; n++) {
    if (!trace_step(a.g, og, icell, xe, ye, ze, t)) return 1;
    step(t);
    bool valid = true;
#pragma unroll
    for (int c = 0; c < 4; c++) valid = valid && ((a.preset[t.i[c]] & presetbit) || rank[t.i[c]] < rp);
    if (valid) return 0;
    if (t.next < 0) return 2;
    icell = t.next;
  }
  return 8;
}

__device__ inline int chain_count(const SweepArgs& a, int o) {
  return a.lvl_off[a.lo_base[o] + a.nlev[o]] - a.lvl_off[a.lo_base[o]];
}

// The corners each characteristic stops on, by the octant's list order (a
// topological order of every ordinate of the octant).
__global__ __launch_bounds__(256) void k_chain_corners(SweepArgs a, ChainArrays c) {
  const int col = blockIdx.y, j = blockIdx.x * 256 + threadIdx.x;
  const int o = a.col_oct[col];
  if (j >= chain_count(a, o)) return;
  const int e = a.lvl_off[a.lo_base[o]] + j, code = a.lvl_pts[e], pt = code >= 0 ? code : ~code;
  const OrdGeom og = a.ordg[col];
  TraceStep t;
  const int bad = chain_walk(a, og, o, pt, a.lvl_cell[e], t, [](const TraceStep&) {});
  // a bad trace reads itself; k_chain_source reports it
  ushort4 q = make_ushort4(pt, pt, pt, pt);
  if (!bad) q = make_ushort4(t.i[0], t.i[1], t.i[2], t.i[3]);
  c.q[(size_t)col * a.npts + j] = q;
}

// Levels of one ordinate's points (1 + the largest of its corners'), and the
// points in (level) order.  One wavefront takes the list 64 entries at a time;
// few of them read each other, so a chunk settles in a few LDS round trips.
__global__ __launch_bounds__(64) void k_chain_levels(SweepArgs a, ChainArrays c) {
  extern __shared__ uint16_t lev[];
  const int col = blockIdx.x, lane = threadIdx.x;
  const int o = a.col_oct[col], n = chain_count(a, o);
  const int32_t* pts = a.lvl_pts + a.lvl_off[a.lo_base[o]];
  const size_t row = (size_t)col * a.npts;
  int* cnt = c.count + (size_t)col * (a.npts + 2);
  for (int i = lane; i < a.npts; i += 64) lev[i] = 0;
  for (int i = lane; i < a.npts + 2; i += 64) cnt[i] = 0;
  __syncthreads();
  int top = 0;
  for (int j0 = 0; j0 < n; j0 += 64) {
    const int j = min(j0 + lane, n - 1);
    const uint2 q = reinterpret_cast<const uint2*>(c.q)[row + j];
    const int code = pts[j], pt = code >= 0 ? code : ~code;
    // entries of one chunk may read each other: repeat until nothing changes
    // (at most 64 times: the list is a topological order)
    int l = 0;
    for (int it = 0; it < 65; it++) {
      // (a bad trace reads itself and would climb with every turn: no level is
      // past the number of entries, which the counts and the row are sized for)
      const int m = min(n, 1 + max(max((int)lev[q.x & 0xffff], (int)lev[q.x >> 16]),
                                   max((int)lev[q.y & 0xffff], (int)lev[q.y >> 16])));
      const bool changed = m != l;
      l = m;
      if (!__any(changed)) break;
      lev[pt] = (uint16_t)l;
      wave_lds_fence();
    }
    top = max(top, l);
  }
  for (int d = 32; d > 0; d >>= 1) top = max(top, __shfl_xor(top, d));
  __syncthreads();
  for (int j = lane; j < n; j += 64) {
    const int code = pts[j];
    atomicAdd(cnt + lev[code >= 0 ? code : ~code], 1);
  }
  __syncthreads();
  // exclusive prefix sum of the counts: each level's first position
  int base = 0;
  for (int l0 = 1; l0 <= top; l0 += 64) {
    const int l = l0 + lane;
    const int v = l <= top ? atomicAdd(cnt + l, 0) : 0;
    int s = v;
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(s, d);
      if (lane >= d) s += u;
    }
    if (l <= top) atomicExch(cnt + l, base + s - v);
    base += __shfl(s, 63);
  }
  __syncthreads();
  for (int j = lane; j < n; j += 64) {
    const int code = pts[j], l = lev[code >= 0 ? code : ~code];
    const int pos = atomicAdd(cnt + l, 1);
    c.order[row + pos] = j;
    c.ptlev[row + pos] = (uint32_t)(code >= 0 ? code : ~code) | (uint32_t)l << 16;
  }
}

// The records in level order: point, corners, the last face's weights and the
// transmission of the whole path.
__global__ __launch_bounds__(256) void k_chain_records(SweepArgs a, ChainArrays c) {
#pragma clang fp contract(off)
  const int col = blockIdx.y, pos = blockIdx.x * 256 + threadIdx.x;
  const int o = a.col_oct[col];
  if (pos >= chain_count(a, o)) return;
  const size_t r = (size_t)col * a.npts + pos;
  const int e = a.lvl_off[a.lo_base[o]] + c.order[r], code = a.lvl_pts[e], pt = code >= 0 ? code : ~code;
  const OrdGeom og = a.ordg[col];
  double ext1 = a.ext[pt], transmit = 1.0;
  TraceStep t;
  const int bad = chain_walk(a, og, o, pt, a.lvl_cell[e], t, [&](const TraceStep& s) {
    const double f1 = (1 - s.u) * (1 - s.v), f2 = (1 - s.u) * s.v, f3 = s.u * (1 - s.v), f4 = s.u * s.v;
    const double ext0 = f1 * a.ext[s.i[0]] + f2 * a.ext[s.i[1]] + f3 * a.ext[s.i[2]] + f4 * a.ext[s.i[3]];
    double src, absc, trc;
    cell_integral(ext0, ext1, 0.0, 0.0, s.so, src, absc, trc);
    transmit = transmit * trc;
    ext1 = ext0;
  });
  c.q[r] = bad ? make_ushort4(pt, pt, pt, pt) : make_ushort4(t.i[0], t.i[1], t.i[2], t.i[3]);
  c.u[r] = bad ? 0.0 : t.u;
  c.v[r] = bad ? 0.0 : t.v;
  c.trans[r] = bad ? 0.0 : transmit;
}

// The source integral of every characteristic, in level order.  Gathers of the
// ordinate's source row (18 KB at 16^3, cache resident); bound by the latency
// of a trace, hidden by the number of them (0.4 M at 16^3 NMU 8).
__global__ __launch_bounds__(256) void k_chain_source(SweepArgs a, ChainArrays c, int col0) {
#pragma clang fp contract(off)
  if (a.stop && *a.stop) return;
  const int col = col0 + blockIdx.y, kst = blockIdx.z, pos = blockIdx.x * 256 + threadIdx.x;
  const int o = a.col_oct[col];
  if (pos >= chain_count(a, o)) return;
  const size_t r = (size_t)col * a.npts + pos;
  const int e = a.lvl_off[a.lo_base[o]] + c.order[r], code = a.lvl_pts[e], pt = code >= 0 ? code : ~code;
  const OrdGeom og = a.ordg[col];
  const float* se = a.srcext + kst * a.pdo + (size_t)col * a.ldp;
  double ext1 = a.ext[pt], srcext1 = se[pt], radv = 0.0, transmit = 1.0;
  TraceStep t;
  const int bad = chain_walk(a, og, o, pt, a.lvl_cell[e], t, [&](const TraceStep& s) {
    const double f1 = (1 - s.u) * (1 - s.v), f2 = (1 - s.u) * s.v, f3 = s.u * (1 - s.v), f4 = s.u * s.v;
    const double ext0 = f1 * a.ext[s.i[0]] + f2 * a.ext[s.i[1]] + f3 * a.ext[s.i[2]] + f4 * a.ext[s.i[3]];
    const double srcext0 = f1 * se[s.i[0]] + f2 * se[s.i[1]] + f3 * se[s.i[2]] + f4 * se[s.i[3]];
    double src, absc, trc;
    cell_integral(ext0, ext1, srcext0, srcext1, s.so, src, absc, trc, kst == 0);
    radv = radv + transmit * src * absc;
    transmit = transmit * trc;
    ext1 = ext0;
    srcext1 = srcext0;
  });
  if (bad) atomicOr(a.errflag, bad);
  // the list the levels were made in is the host planner's: every corner
  // computed in the sweep lies on a lower one of its levels
  const int32_t* level = a.level + (size_t)o * a.npts;
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (!bad && !(a.preset[t.i[k]] & (og.bitz ? 2 : 1)) && level[t.i[k]] >= level[pt]) atomicOr(a.errflag, 4);
  c.radv[kst * c.plane + r] = bad ? 0.0 : radv;
}

constexpr int CHAIN_THREADS = 256;
constexpr int CHAIN_F64_POINTS = 20480;   // a row of doubles fits in 160 KB
constexpr int CHAIN_AHEAD = 6;   // chunks of 64 records in flight

// One ordinate's radiances in level order.  The first wavefront runs the
// chain, 64 records at a time (one per lane, the next CHAIN_AHEAD chunks loading
// meanwhile): the lanes of one level gather their corners from the LDS row and write their
// points, then the next level's lanes do; a wavefront's LDS operations are in
// order, so levels need no barrier, only a fence for the compiler.  Bound by levels x (LDS round trip + the
// FP64 sum).  The row is kept in doubles where they fit (four conversions less
// per level: 0.29 against 0.33 ms at 16^3 periodic).  The other wavefronts help
// to fill and write out the row.
template <typename Row>
__global__ __launch_bounds__(CHAIN_THREADS) void k_sweep_chain(SweepArgs a, ChainArrays c, int col0) {
  if (a.stop && *a.stop) return;
  extern __shared__ double row_lds[];
  Row* row = reinterpret_cast<Row*>(row_lds);
  const int col = col0 + blockIdx.x, kst = blockIdx.y, tid = threadIdx.x;
  const int o = a.col_oct[col], n = chain_count(a, o);
  const int up = (o >> 2) & 1;
  const int nbc = up ? a.nbot : a.ntop;
  const int32_t* bc = up ? a.bcbot : a.bctop;
  for (int b = tid; b < nbc; b += CHAIN_THREADS) row[bc[b]] = kst ? 0.0f : up ? a.bcrad_bot[b] : a.skyrad[col];
  __syncthreads();
  if (tid < 64 && n > 0) {
    const size_t r0 = (size_t)col * a.npts;
    const uint2* gq = reinterpret_cast<const uint2*>(c.q) + r0;
    const double* gr = c.radv + kst * c.plane + r0;
    struct Rec {
      uint2 q;
      double u, v, t, r;
      uint32_t ptlev;
    };
    // (past the end: the last record again, never run)
    auto load = [&](int p0, Rec& x) {
      const int p = min(p0 + tid, n - 1);
      x.q = gq[p];
      x.u = c.u[r0 + p];
      x.v = c.v[r0 + p];
      x.t = c.trans[r0 + p];
      x.r = gr[p];
      x.ptlev = c.ptlev[r0 + p];
    };
    auto run = [&](int p0, const Rec& x) {
      if (p0 >= n) return;
      const double tu = x.t * x.u, t1 = x.t - tu;
      const double f1 = t1 * (1 - x.v), f2 = t1 * x.v, f3 = tu * (1 - x.v), f4 = tu * x.v;
      const Row *q1 = row + (x.q.x & 0xffff), *q2 = row + (x.q.x >> 16);
      const Row *q3 = row + (x.q.y & 0xffff), *q4 = row + (x.q.y >> 16);
      Row* out = row + (x.ptlev & 0xffff);
      const int lev = p0 + tid < n ? (int)(x.ptlev >> 16) : 0;
      const int l0 = __builtin_amdgcn_readlane(lev, 0), l1 = __builtin_amdgcn_readlane(lev, min(n - p0, 64) - 1);
      for (int l = l0; l <= l1; l++) {
        if (lev == l) {
          const double r1 = *q1, r2 = *q2, r3 = *q3, r4 = *q4;
          *out = (float)(fma(f2, r2, fma(f1, r1, x.r)) + fma(f4, r4, f3 * r3));
        }
        wave_lds_fence();
      }
    };
    Rec x[CHAIN_AHEAD];
#pragma unroll
    for (int k = 0; k < CHAIN_AHEAD; k++) load(k * 64, x[k]);
    for (int p0 = 0; p0 < n; p0 += CHAIN_AHEAD * 64) {
#pragma unroll
      for (int k = 0; k < CHAIN_AHEAD; k++) {
        run(p0 + k * 64, x[k]);
        load(p0 + (k + CHAIN_AHEAD) * 64, x[k]);
      }
    }
  }
  __syncthreads();
  float* rad = a.rad + kst * a.pdo + (size_t)col * a.ldp;
  for (int i = tid; i < a.npts; i += CHAIN_THREADS) rad[i] = (float)row[i];
}

static bool chain_row_f64(int npts) { return npts <= CHAIN_F64_POINTS; }

int sweep_chain_max_lds(int npts) {
  const void* k = chain_row_f64(npts) ? reinterpret_cast<const void*>(k_sweep_chain<double>)
                                      : reinterpret_cast<const void*>(k_sweep_chain<float>);
  return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, npts * (chain_row_f64(npts) ? 8 : 4)) ==
                 hipSuccess &&
                 hipFuncSetAttribute(reinterpret_cast<const void*>(k_chain_levels),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, npts * 2) == hipSuccess
             ? 0
             : 1;
}

void launch_chain_setup(hipStream_t st, const SweepArgs& a, const ChainArrays& c, int ncol) {
  const dim3 grid((a.npts + 255) / 256, ncol);
  k_chain_corners<<<grid, 256, 0, st>>>(a, c);
  k_chain_levels<<<ncol, 64, (size_t)a.npts * 2, st>>>(a, c);
  k_chain_records<<<grid, 256, 0, st>>>(a, c);
}

void launch_sweep_chain(hipStream_t st, const SweepArgs& a, const ChainArrays& c, int col0, int ncol) {
  if (ncol <= 0) return;
  k_chain_source<<<dim3((a.npts + 255) / 256, ncol, a.nst), 256, 0, st>>>(a, c, col0);
  const dim3 grid(ncol, a.nst);
  if (chain_row_f64(a.npts))
    k_sweep_chain<double><<<grid, CHAIN_THREADS, (size_t)a.npts * 8, st>>>(a, c, col0);
  else
    k_sweep_chain<float><<<grid, CHAIN_THREADS, (size_t)a.npts * 4, st>>>(a, c, col0);
}

}  // namespace at3d
