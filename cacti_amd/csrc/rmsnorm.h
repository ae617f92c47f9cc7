// The RMSNorm adjoint in two parts (rmsnorm.hip): the input's gradient with partial rows of the weight's, and the sums of such
// rows, of several norms in one launch.
#pragma once
#include "common.h"

namespace cacti {

constexpr int kRmsNormDwSums = 16;            // norms of a launch
// cacti_hip_rms_norm_bwd without the sum: part [G][D] fp32, cacti_hip_rms_norm_bwd_workspace(N, D) bytes
int rms_norm_bwd_parts(int64_t N, int64_t D, const void *x, const void *w, float eps, const void *dy, void *dx, int dx_acc, void *part,
                       size_t part_bytes, hipStream_t st);
// dw[i][D] (+)= f16 of the sum of the rows of part[i] [G][D], in the same order as cacti_hip_rms_norm_bwd; bit i of acc: added to
int rms_norm_dw_sums(int n, int64_t G, int64_t D, const void *const *part, void *const *dw, uint32_t acc, hipStream_t st);

}  // namespace cacti
