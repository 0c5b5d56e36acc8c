// The affine map z = y a + b of a batch norm channel, for the kernels that make it: from the statistics of a batch
// (bn_finalize_kernel) or from the running ones (there, or in the launch that prepares the convolution's weights).
#pragma once

#include "sjhip_common.h"

namespace sjhip {

// Evaluation mode: where the running statistics lie and where the map goes ([4][C]: a, b, mean, 1/std).
struct BnEvalMap {
  const float *gamma, *beta, *running_mean, *running_var;
  float eps;
  float *map;  // nullptr: no map asked for
  int C;
};

#ifdef __HIPCC__
__device__ __forceinline__ void store_bn_map(int c, double mean, double var, const float *gamma, const float *beta, float eps,
                                             float *scale, float *shift, float *mean_out, float *invstd_out) {
  const double invstd = 1.0 / sqrt(var + (double)eps);
  const double g = gamma ? (double)gamma[c] : 1.0, b = beta ? (double)beta[c] : 0.0;
  const double a = g * invstd;
  scale[c] = (float)a;
  shift[c] = (float)(b - mean * a);
  mean_out[c] = (float)mean;
  invstd_out[c] = (float)invstd;
}
__device__ __forceinline__ void store_bn_map(const BnEvalMap &e, int c) {
  store_bn_map(c, (double)e.running_mean[c], (double)e.running_var[c], e.gamma, e.beta, e.eps, e.map, e.map + e.C, e.map + 2 * e.C, e.map + 3 * e.C);
}
#endif

// launch_pwconv_split_weight_f16 of W [rows][cols] that also makes the map of the batch norm behind the convolution
int launch_pwconv_split_weight_f16_bn(const float *w, int64_t rows, int64_t cols, uint16_t *planes, float *amax_reset,
                                      int64_t amax_floats, const BnEvalMap &bn, hipStream_t stream);

}  // namespace sjhip
