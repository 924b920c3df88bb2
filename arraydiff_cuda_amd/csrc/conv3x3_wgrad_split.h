// The filter gradient of the 3x3 window at stride 1 in fp32: what conv3x3_wgrad_split.hip gives the entry points.
#ifndef ADH_CONV3X3_WGRAD_SPLIT_H
#define ADH_CONV3X3_WGRAD_SPLIT_H

#include "adh_common.h"

namespace adh {

// dw[co][ci][a][b] = beta*dw + sum over images, R, Q of dy[co][R][Q] * x[ci][R + a - pad_r][Q + b - pad_c] (zero outside x)
struct Wgrad3x3Problem {
  uint32_t num_tiles, N, Cin, Cout;
  uint32_t x_H, x_W, dy_H, dy_W;
  // stacked: the tiles are the row tiles of one tensor in rank order and carry no halo.  neighbours: they carry one halo row
  // above and below whose inner ones are to be read from the neighbouring tiles' interiors; the sums are then taken tile by
  // tile as if the halos had been exchanged (the same bits).  Neither: every tile is a tensor of its own.
  bool stacked, neighbours;
  int32_t pad_r, pad_c;
  const void *const *x, *const *dy;
  float *dw;
  float beta;
};

// enough for every form (padded, unexchanged, without halo) of the layer whose tiles' interiors are H x W
size_t conv3x3_wgrad_split_workspace(uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W);
// the least that it runs with: in a smaller workspace than the above the pixels are dealt to fewer workgroups, below a workgroup
// per channel group the groups are launched in turn
size_t conv3x3_wgrad_split_least_workspace(uint32_t Cin, uint32_t Cout);
int conv3x3_wgrad_split(const Wgrad3x3Problem &q, void *workspace, size_t workspace_bytes, hipStream_t st);

}  // namespace adh
#endif
