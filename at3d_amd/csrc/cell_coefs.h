// The cell integral of a short characteristic in single precision, and the
// workgroup barrier and wavefront fence of the sweeps (device).
#pragma once
#include <hip/hip_runtime.h>

namespace at3d {

// Barrier that orders LDS traffic only: outstanding global loads (the next
// levels' records) and stores (radiances) stay in flight across it.
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Orders a wavefront's own LDS traffic: what its lanes wrote before is what its
// other lanes read after.  The hardware keeps a wavefront's LDS operations in
// order, so no instruction comes of it; without it nothing keeps the compiler
// from moving one lane's load over another's store.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// 1 / x to a last place: the hardware's estimate and one Newton step (3
// instructions against the 10 of a correctly rounded division).
__device__ inline float recip(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.0f), r, r);
}

// The cell integral of a one-cell step (shdomsub1.f:3948-3987, with the
// reference's tau branches) as coefficients of the face and point sources:
// src x abs = b0 SRCEXT0 + b1 SRCEXT1 before the clamp at zero, and the
// cell's transmission, in single precision from the face and point
// extinctions and the path length.
__device__ inline void cell_coefs(float ext0, float ext1, float so, float& b0, float& b1, float& trc) {
  const float e = 0.5f * (ext0 + ext1);
  const float tau = e * so;
  float absc;
  if (tau >= 0.5f) {
    trc = __expf(-tau);
    absc = 1.0f - trc;
  } else {
    absc = tau * (1.0f - 0.5f * tau * (1.0f - 0.33333333333f * tau * (1.0f - 0.25f * tau)));
    trc = 1.0f - absc;
  }
  float c0, c1;
  if (tau <= 2.0f) {
    // (e = 0: absc is 0, and so are b0 and b1)
    const float k = 0.08333333333f * so, re = __builtin_amdgcn_rcpf(fmaxf(e, 1e-30f));
    c0 = (0.5f - k * ext1) * re;
    c1 = (0.5f + k * ext0) * re;
  } else {
    float e0p = ext0, sc = 1.0f;
    if (tau > 4.0f) {
      e0p = ext1 + (ext0 - ext1) * 4.0f * recip(tau);
      if (ext0 > 0.0f) sc = e0p * recip(ext0);
    }
    const float rd = recip(e0p + ext1);
    const float g = 2.0f * rd * (1.0f - 2.0f * recip(tau) + 2.0f * trc * recip(absc));
    c0 = sc * (1.0f - ext1 * g) * rd;
    c1 = (1.0f + e0p * g) * rd;
  }
  b0 = c0 * absc;
  b1 = c1 * absc;
}

}  // namespace at3d
