// DO->SH by factors (DO_TO_SH, shdomsub1.f:3041-3254): the azimuth sums per
// zenith angle, then the Legendre sums per m, as the reference splits them, both
// on the matrix cores.
//
// The dense product (k_do_to_sh) costs NANG x NLM multiply-adds a point, 354 x
// 256 at NMU 16, and every partial sum of 354 terms.  By factors a zenith
// angle's n azimuths fold onto cosine and sine halves (phi and -phi), n^2 / 2
// terms, and a coefficient takes NMU terms: a fifth of the matrix work.
//
// One workgroup per CU takes tiles of 64 columns in turn: 64 points, or 32
// points' Q and U.  In the first step a wavefront takes a zenith angle (A: the
// angle's cosines or sines, m x azimuth; B: folded radiances, azimuth x 16
// columns) and leaves the azimuth sums in LDS; in the second it takes orders m
// (A: weighted Legendre functions, l x zenith angle; B: those sums) and leaves
// the coefficients in LDS, from where they go out as rows.  The next tile's
// radiances fly meanwhile.  Orders that no point of the tile keeps are not
// computed; rows are zero at and past the point's radiance count, and zeros go
// out only where the row's last write left terms (rlen; every other writer of R
// sets it past the end).  Q and U: their Legendre functions are the same up to
// sign, so both components' products share the operands.
//
// Bound by the round trips of a tile with one workgroup on a CU (its LDS holds
// 64 columns' sums and coefficients), at about half the rate of a large copy.  Q
// and U with more than 8 zenith angles spill 2 vector registers up to 31 azimuths,
// 11 from 32 on.
// NMU 16, an iteration, the dense product before: 64 x 64 x 40 81 us for 240,
// 96 x 96 x 48 216 for 645, 128 x 128 x 64 I 0.51 ms for 1.48 and Q with U 1.52
// for 5.40.  Tried: the same sums a lane a point from scalar tables, 170 us at
// 64 x 64 x 40; tiles of 32 columns, two workgroups a CU, 122; the next tile's
// loads issued before the second step's operands (loads return in order), 92.
// Error of R against FP64: 5.5e-8, the dense product's 2e-7 and more.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <numeric>

#include "analysis.h"
#include "cell_coefs.h"
#include "kernels.h"
#include "ring_plan.h"

namespace at3d {

namespace {

typedef float float4_ __attribute__((ext_vector_type(4)));
constexpr int UNIT_INTS = 8;
constexpr int QMAX = 5;    // quads of folded azimuths of a zenith angle
constexpr int ZQ = 4;      // quads of zenith angles
constexpr int CUS = 256;

// WAVES wavefronts, one for each zenith angle; QM quads of azimuths at most.
template <int WAVES, int QM, bool QU>
__global__ __launch_bounds__(64 * WAVES, 4) void k_analysis(const float* __restrict__ D, AnalysisArgs t,
                                                            const int* __restrict__ nr, int* __restrict__ rlen,
                                                            float* __restrict__ R, int nlm, int mm, int ld, int ldp,
                                                            size_t upper, int npts, const int* __restrict__ stop,
                                                            size_t plane) {
  if (stop && *stop) return;
  extern __shared__ float lds[];
  constexpr int TP = QU ? 32 : 64;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, kk = lane >> 4;
  // neighbouring tiles share pages of the radiance rows: each XCD (dealt
  // workgroups round robin, with an L2 of its own) takes a run of them
  const int tiles = (npts + TP - 1) / TP, per = (tiles + 7) / 8, step = gridDim.x / 8;
  int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int end = min(tiles, ((blockIdx.x & 7) + 1) * per);
  if (tile >= end) return;
  // this wavefront's zenith angle: its quads of azimuths, largest m, row of
  // m = 0 in F, columns and A
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  const int32_t* info = t.ints + w * UNIT_INTS;
  const bool has = w < t.nunits;
  const int nq = has ? uniform(info[0]) : 0, me = has ? uniform(info[1]) : 0, row0 = has ? uniform(info[2]) : 0;
  float ac[QM], as[QM];
  if (has) {
    const float* trig = t.floats + uniform(info[3]) + lane;
#pragma unroll
    for (int q = 0; q < QM; q++)
      if (q < nq) {
        ac[q] = trig[q * 128];
        as[q] = trig[q * 128 + 64];
      }
  }
  // this lane's zenith angles: row of m = 0 and largest m
  int zrow[ZQ], zme[ZQ];
#pragma unroll
  for (int q = 0; q < ZQ; q++) {
    const int2 z = reinterpret_cast<const int2*>(t.ints + t.zenith)[4 * q + kk];
    zrow[q] = z.x;
    zme[q] = z.y;
  }
  // columns 4 j + g of a tile: point 4 j + g, or points 2 j and 2 j + 1 of Q,
  // then of U
  const int nzq = t.nzq;
  float* T = lds;                           // [64][ldt] coefficients
  const int ldt = nlm | 1;
  int2* cols = reinterpret_cast<int2*>(lds + 64 * ldt) + w * (4 * QM);   // this angle's columns
  float* F = lds + 64 * ldt + WAVES * (8 * QM);   // [rows][64] azimuth sums
  if (lane < 4 * QM)
    cols[lane] = has ? reinterpret_cast<const int2*>(t.ints + uniform(info[4]))[lane] : make_int2(0, 0);
  lds_barrier();
  float4_ a[QM], b[QM];
  int n_next, was_next;
  // A tile's radiances and radiance counts (of this row write and the last one),
  // in two parts: loads return in order, and only a fixed number of them behind a
  // value lets it be waited for alone.  Quads past nq read the first column again.
  auto get = [&](int p0, int2 c, int q) {
    // (a uniform base and 32-bit byte offsets: one register an address)
    const char *Dp = reinterpret_cast<const char*>(D + p0), *Du = Dp + upper * 4;
    const uint32_t own = (QU ? 8u : 16u) * j, row = (uint32_t)ldp * 4;
    const uint32_t x = (uint32_t)c.x * row + own, y = (uint32_t)c.y * row + own;
    if (QU) {
      const float2 aq = *reinterpret_cast<const float2*>(Dp + x), au = *reinterpret_cast<const float2*>(Du + x);
      const float2 bq = *reinterpret_cast<const float2*>(Dp + y), bu = *reinterpret_cast<const float2*>(Du + y);
      a[q] = (float4_){aq.x, aq.y, au.x, au.y};
      b[q] = (float4_){bq.x, bq.y, bu.x, bu.y};
    } else {
      a[q] = *reinterpret_cast<const float4_*>(Dp + x);
      b[q] = *reinterpret_cast<const float4_*>(Dp + y);
    }
  };
  auto load_counts = [&](int p0) {
    const int i0 = lane < TP && p0 + lane < npts ? p0 + lane : -1;
    n_next = i0 >= 0 ? nr[i0] : 0;
    was_next = i0 >= 0 ? rlen[i0] : 0;
  };
  auto load = [&](int p0) {
#pragma unroll
    for (int q = 0; q < QM; q++) get(p0, cols[4 * q + kk], q);
  };
  load_counts(tile * TP);
  load(tile * TP);
  for (; tile < end; tile += step) {
    const int p0 = tile * TP;
    const int n = n_next, was = was_next;
    // the tile's largest radiance count
    int tile_nr = n;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) tile_nr = max(tile_nr, __shfl_xor(tile_nr, off));
    tile_nr = uniform(tile_nr);
    // largest m of the terms below tile_nr: l (l + 1) + m < tile_nr
    const int mtile = tile_nr > 0 ? min(mm, (int)sqrtf((float)tile_nr - 0.5f)) : -1;
    if (tile_nr > 0 && nq > 0) {
      const int mtop = min(me, mtile);
      float* f = F + row0 * 64 + 4 * j;
      // (two columns at a time: the registers of four spill)
#pragma unroll
      for (int h = 0; h < 4; h += 2) {
        float4_ C[2], S[2];
#pragma unroll
        for (int g = 0; g < 2; g++) C[g] = S[g] = (float4_){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < QM; q++)
          if (q < nq) {
#pragma unroll
            for (int g = 0; g < 2; g++) {
              C[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(ac[q], a[q][h + g] + b[q][h + g], C[g], 0, 0, 0);
              S[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(as[q], a[q][h + g] - b[q][h + g], S[g], 0, 0, 0);
            }
          }
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int m = 4 * kk + v;
          if (m <= mtop) {
            // m > 0: cos - sin, m < 0: cos + sin (m = 0: no sine)
            *reinterpret_cast<float2*>(f + m * 64 + h) = make_float2(C[0][v] - S[0][v], C[1][v] - S[1][v]);
            *reinterpret_cast<float2*>(f - m * 64 + h) = make_float2(C[0][v] + S[0][v], C[1][v] + S[1][v]);
          }
        }
      }
    }
    // the second step's A before the next tile's radiances (the last tile's again;
    // addresses made anew for each tile: kept ones spill)
    const int next = tile + step < end ? tile + step : tile;
    load_counts(next * TP);
    __builtin_amdgcn_sched_barrier(0);
    int la = lane;
    asm volatile("" : "+v"(la));
    const int ja = la & 15, ka = la >> 4;
    float A[2][ZQ], X[2][ZQ];
#pragma unroll
    for (int turn = 0; turn < 2; turn++) {
      const int am = min(mm, (w + turn * WAVES + 1) >> 1);
      const float* leg = t.floats + t.legendre + am * (ZQ * 64 * (QU ? 2 : 1)) + la;
#pragma unroll
      for (int q = 0; q < ZQ; q++) {
        A[turn][q] = leg[q * 64];
        if (QU) X[turn][q] = leg[(ZQ + q) * 64];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    load(next * TP);
    __builtin_amdgcn_sched_barrier(0);
    if (tile_nr > 0) {
      lds_barrier();
#pragma unroll
      for (int turn = 0; turn < 2; turn++) {
        const int c = w + turn * WAVES, am = (c + 1) >> 1, m = c & 1 ? am : -am;
        if (c >= 2 * mtile + 1) continue;
        float4_ acc[4];
#pragma unroll
        for (int g = 0; g < 4; g++) acc[g] = (float4_){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < ZQ; q++)
          if (q < nzq) {
            // (an angle without this m has a zero in A; its last row stands in)
            const int mz = max(-zme[q], min(zme[q], m));
            const float* f = F + 4 * ja + (zrow[q] + mz) * 64;
            if (QU) {
              const float s = m < 0 ? -1.f : 1.f;
              const float2 fq = *reinterpret_cast<const float2*>(f);
              const float2 u = *reinterpret_cast<const float2*>(f - 128 * mz + 2);
              const float2 fu = make_float2(s * u.x, s * u.y);
              acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[turn][q], fq.x, acc[0], 0, 0, 0);
              acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[turn][q], fq.y, acc[1], 0, 0, 0);
              acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[turn][q], fu.x, acc[2], 0, 0, 0);
              acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[turn][q], fu.y, acc[3], 0, 0, 0);
              acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(X[turn][q], fu.x, acc[0], 0, 0, 0);
              acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(X[turn][q], fu.y, acc[1], 0, 0, 0);
              acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(X[turn][q], fq.x, acc[2], 0, 0, 0);
              acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(X[turn][q], fq.y, acc[3], 0, 0, 0);
            } else {
              const float4_ x = *reinterpret_cast<const float4_*>(f);
#pragma unroll
              for (int g = 0; g < 4; g++)
                acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[turn][q], x[g], acc[g], 0, 0, 0);
            }
          }
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int l = am + 4 * ka + v;
          const int J = (l <= mm ? l * (l + 1) : (2 * mm + 1) * l - mm * mm) + m;
          if (J < tile_nr) {
#pragma unroll
            for (int g = 0; g < 4; g++) T[(4 * ja + g) * ldt + J] = acc[g][v];
          }
        }
      }
      lds_barrier();
    }
    // the rows, zeros up to where the last write's terms ended
    for (int r = w; r < 64; r += WAVES) {
      const int i = QU ? 2 * (r >> 2) + (r & 1) : r;
      if (p0 + i >= npts) continue;
      const bool second = QU && (r & 2);
      const int nq = __builtin_amdgcn_readlane(n, i), top = min(ld, max(nq, __builtin_amdgcn_readlane(was, i)));
      float* out = R + (size_t)(p0 + i) * ld + (second ? plane : 0);
      for (int x = lane; x < top; x += 64) out[x] = x < nq ? T[r * ldt + x] : 0.f;
      if (lane == 0 && !second) rlen[p0 + i] = nq;
    }
  }
}

template <int WAVES, int QM, bool QU>
void go(int grid, size_t lds, hipStream_t st, const float* D, const AnalysisArgs& t, const int* nr, int* rlen, float* R,
        int nlm, int mm, int ld, int ldp, size_t upper, int npts, const int* stop, size_t plane) {
  k_analysis<WAVES, QM, QU><<<grid, 64 * WAVES, lds, st>>>(D, t, nr, rlen, R, nlm, mm, ld, ldp, upper, npts, stop, plane);
}

// By zenith angles (a wavefront each, two orders m each) and azimuths.
struct Shape {
  int waves, quads;
  const void* f[2];   // scalar, Q and U
  decltype(&go<8, 3, false>) run[2];
};
template <int WAVES, int QM>
Shape shape() {
  return {WAVES, QM,
          {reinterpret_cast<const void*>(k_analysis<WAVES, QM, false>), reinterpret_cast<const void*>(k_analysis<WAVES, QM, true>)},
          {go<WAVES, QM, false>, go<WAVES, QM, true>}};
}
const Shape* shape_of(const Plan& p) {
  static const Shape shapes[] = {shape<8, 3>(), shape<16, 4>(), shape<16, QMAX>()};
  const int n0 = *std::max_element(p.nphi0.begin(), p.nphi0.end());
  for (const Shape& s : shapes)
    if (p.nmu <= s.waves && p.mm < s.waves && n0 / 2 + 1 <= 4 * s.quads) return &s;
  return nullptr;
}

}  // namespace

// (32-bit byte offsets into a Stokes component's radiances)
bool analysis_takes(const Plan& p) {
  return p.nmu <= 4 * ZQ && p.ml <= 15 && p.mm <= p.ml && shape_of(p) &&
         (uint64_t)(p.nang + 63) * (p.npts + 64) * 4 < (1ull << 32);
}

bool build_analysis(const Plan& p, const std::vector<int32_t>& col_of_ref, bool qu, AnalysisTables& t) {
  t = AnalysisTables();
  if (!analysis_takes(p)) return false;
  const int nmu = p.nmu, nlm = p.nlm;
  std::vector<int> first(nmu, 0), row0(nmu, 0), me(nmu, 0), order(nmu);
  int rows = 0;
  for (int i = 0; i < nmu; i++) {
    first[i] = i ? first[i - 1] + p.nphi0[i - 1] : 0;
    me[i] = std::max(0, std::min(p.nphi0[i] / 2 - 1, p.mm));
    row0[i] = rows + me[i];   // of m = 0
    rows += 2 * me[i] + 1;
  }
  // zenith angles, most azimuths first
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return p.nphi0[a] > p.nphi0[b]; });
  std::vector<int32_t>& I = t.ints;
  std::vector<float>& F = t.floats;
  I.assign(nmu * UNIT_INTS, 0);
  t.a.nunits = nmu;
  for (int u = 0; u < nmu; u++) {
    const int i = order[u], n0 = p.nphi0[i], nk = n0 / 2 + 1, nq = (nk + 3) / 4;
    const int32_t info[5] = {nq, me[i], row0[i], (int32_t)F.size(), (int32_t)I.size()};
    std::copy(info, info + 5, I.begin() + u * UNIT_INTS);
    for (int k = 0; k < 4 * shape_of(p)->quads; k++) {
      const int k1 = k < nk ? k : 0;
      I.push_back(col_of_ref[first[i] + k1]);
      I.push_back(col_of_ref[first[i] + (n0 - k1) % n0]);
    }
    // A[m][k]: lane m + 16 (k % 4); phi = 0 and pi are their own images
    const double dphi = 2.0 * acos(-1.0) / n0;
    for (int q = 0; q < nq; q++)
      for (int sine = 0; sine < 2; sine++)
        for (int lane = 0; lane < 64; lane++) {
          const int m = lane & 15, k = 4 * q + (lane >> 4);
          const bool self = (n0 - k) % n0 == k;
          const double x = (double)((m * k) % n0) * dphi;
          const double v = sine ? (self ? 0.0 : sin(x)) : (self ? 0.5 * cos(x) : cos(x));
          F.push_back(k < nk && m <= me[i] ? (float)v : 0.f);
        }
  }
  t.a.nzq = (nmu + 3) / 4;
  t.a.zenith = (int)I.size();
  for (int i = 0; i < 4 * ZQ; i++) {
    I.push_back(row0[std::min(i, nmu - 1)]);
    I.push_back(me[std::min(i, nmu - 1)]);
  }
  // weighted Legendre functions, A[l - |m|][zenith angle]: the tables at phi = 0,
  // where every azimuth factor is one.  Q and U: element 2 for a component's own
  // sums, 6 for the other's (m < 0: signs in the kernel).
  t.a.legendre = (int)F.size();
  for (int am = 0; am <= p.mm; am++)
    for (int e = 0; e < (qu ? 2 : 1); e++)
      for (int q = 0; q < ZQ; q++)
        for (int lane = 0; lane < 64; lane++) {
          const int l = am + (lane & 15), i = 4 * q + (lane >> 4);
          if (l > p.ml || i >= nmu || am > me[i]) {
            F.push_back(0.f);
            continue;
          }
          const int J = (l <= p.mm ? l * (l + 1) : (2 * p.mm + 1) * l - p.mm * p.mm) + am;
          F.push_back(qu ? p.wpol[((size_t)(e ? 5 : 1) * p.nang + first[i]) * nlm + J]
                         : p.wmat[(size_t)first[i] * nlm + J]);
        }
  const Shape* shape = shape_of(p);
  t.shape = shape;
  t.f = shape->f[qu];
  t.lds = (size_t)(64 * (nlm | 1) + shape->waves * 8 * shape->quads + rows * 64) * 4;
  return t.lds <= (size_t)GFX950_LDS_BYTES;
}

int analysis_max_lds(const AnalysisTables& t) {
  return hipFuncSetAttribute(t.f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)t.lds) == hipSuccess ? 0 : 1;
}

void launch_analysis(hipStream_t st, const AnalysisTables& t, bool qu, const float* dorad, const int* nr, int* rlen,
                     float* R, int nlm, int mm, int ld, int ldo, int ldp, int npts, const int* stop,
                     size_t plane) {
  const Shape& s = *static_cast<const Shape*>(t.shape);
  const int tp = qu ? 32 : 64, tiles = (npts + tp - 1) / tp, groups = CUS * 16 / s.waves;
  s.run[qu](std::min((tiles + 7) / 8 * 8, groups), t.lds, st, dorad, t.a, nr, rlen, R, nlm, mm, ld, ldp,
            (size_t)ldo * ldp, npts, stop, plane);
}

}  // namespace at3d
