// Convolution of an input with at most three channels on the bf16 matrix cores (conv_thin_split.hip).
#ifndef ADH_CONV_THIN_SPLIT_H
#define ADH_CONV_THIN_SPLIT_H

#include "adh_common.h"

namespace adh {

// fp32, halo-padded tiles of HP x WP, no dilation
struct ThinProblem {
  uint32_t num_tiles, N, Cin, Cout, HP, WP, OH, OW, kh, kw, sh, sw;
  const void *const *x;  // tiles
};

// y = beta*y + conv + bias (null: none).  ADH_EUNIMPL: not a shape this serves; nothing launched.
int conv_thin_split_fwd(const ThinProblem &q, const void *w, void *const *y_tiles, float beta, const float *const *bias_tiles,
                        hipStream_t st);
// bytes of partial sums (0: not a shape this serves), and dw = beta*dw + the filter gradient (in a smaller workspace by fewer
// workgroups; ADH_EUNIMPL: nor does it hold the sums of one)
size_t conv_thin_split_wgrad_workspace(const ThinProblem &q);
int conv_thin_split_wgrad(const ThinProblem &q, const void *const *dy_tiles, float *dw, float beta, void *workspace,
                          size_t workspace_bytes, hipStream_t st);

}  // namespace adh
#endif
