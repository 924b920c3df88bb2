// Filter gradients of 3x3 windows at stride 1 over bf16 tensors, dw in fp32: what conv3x3_wgrad_steps.hip gives the entry points.
#ifndef ADH_CONV3X3_WGRAD_STEPS_H
#define ADH_CONV3X3_WGRAD_STEPS_H

#include "adh_common.h"

namespace adh {

// dw[co][ci][a][b] = beta*dw + sum over images, h, w of dy[co][h][w] * x[ci][h + a][w + b], x with a halo of one (H + 2 x W + 2, tiles of
// their own), or (stacked) x[ci][h + a - 1][w + b - 1] with zeros outside, the tiles being the row tiles of one tensor in rank order.
struct StepsWgradProblem {
  bool stacked;
  uint32_t num_tiles, N, Cin, Cout, H, W;
  const void *const *x, *const *dy;
  float *dw;
  float beta;
};

// as much as it has use for (0: a shape it does not take); it runs with less, down to a workgroup's sums per 64 x 64 channels
size_t conv3x3_wgrad_steps_workspace(const StepsWgradProblem &q);
// expected time (0: a shape it does not take)
double conv3x3_wgrad_steps_us(const StepsWgradProblem &q);
// ADH_EUNIMPL: nothing launched, rows of fewer than eight values or a workspace below the least
int conv3x3_wgrad_steps(const StepsWgradProblem &q, void *workspace, size_t workspace_bytes, hipStream_t st);

}  // namespace adh
#endif
