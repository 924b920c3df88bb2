// Filter gradients at stride 2 over tiles without halo: what conv_s2_wgrad.hip gives the entry points.
#ifndef ADH_CONV_S2_WGRAD_H
#define ADH_CONV_S2_WGRAD_H

#include "adh_common.h"

namespace adh {

// dw[co][ci][a][b] = beta*dw + sum over images, R, Q of dy[co][R][Q] * x[ci][2R + a - 1][2Q + b - 1], a 3x3 window with padding 1
// (taps 9), or x[ci][2R][2Q], a 1x1 window (taps 1).  The tiles are the row tiles of one tensor in rank order, dy_H x dy_W and
// 2 dy_H x 2 dy_W; fp32 or bf16 (dtype), dw in fp32.
struct S2WgradProblem {
  int dtype, taps;
  uint32_t num_tiles, N, Cin, Cout, dy_H, dy_W;
  const void *const *x, *const *dy;
  float *dw;
  float beta;
};

// as much as it has use for (0: a shape it does not take); it runs with less, down to a workgroup's sums per 64 x 64 channels
size_t conv_s2_wgrad_workspace(const S2WgradProblem &q);
// what a call has to bring in fp32 (3x3): the sums of 64 x 32 channels' workgroups over chunks of 32 pixels, two workgroups per
// compute unit and at least four chunks each
size_t conv_s2_wgrad_required(const S2WgradProblem &q);
// ADH_EUNIMPL: nothing launched, rows of fewer than four outputs or a workspace below the least
int conv_s2_wgrad(const S2WgradProblem &q, void *workspace, size_t workspace_bytes, hipStream_t st);

}  // namespace adh
#endif
