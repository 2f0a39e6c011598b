// DO->SH by azimuth and Legendre sums (analysis.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "host_plan.h"

namespace at3d {

// Tables on the device and the places of their parts.
struct AnalysisArgs {
  const int32_t* ints = nullptr;
  const float* floats = nullptr;
  int nunits = 0, nzq = 0, zenith = 0, legendre = 0;
};

struct AnalysisTables {
  std::vector<int32_t> ints;   // host copies, for the upload
  std::vector<float> floats;
  AnalysisArgs a;
  const void* f = nullptr;     // the kernel
  size_t lds = 0;
  const void* shape = nullptr; // its launch
};

// Tables of a plan's angle set by device column; qu: of the polarized Q and U.
// False where the angle set has more zenith angles, azimuths or coefficients
// than the kernel takes.
bool analysis_takes(const Plan& p);   // by the sizes alone
bool build_analysis(const Plan& p, const std::vector<int32_t>& col_of_ref, bool qu, AnalysisTables& t);
int analysis_max_lds(const AnalysisTables& t);
// R of npts points from ordinate-major radiances (rows ldp long; U rows ldo rows
// after Q's, R_U `plane` floats after R_Q).  R's rows are zero from rlen on,
// before and after.
void launch_analysis(hipStream_t st, const AnalysisTables& t, bool qu, const float* dorad, const int* nr, int* rlen,
                     float* R, int nlm, int mm, int ld, int ldo, int ldp, int npts, const int* stop,
                     size_t plane);

}  // namespace at3d
