// Windows of 3x3 and 1x1 on bf16 tensors from patches in LDS: what conv_bf16_patch.hip gives the entry points.
#ifndef ADH_CONV_BF16_PATCH_H
#define ADH_CONV_BF16_PATCH_H

#include "conv3x3_split.h"

namespace adh {

// The problem of Conv3x3Problem over bf16 tensors, whose results are rounded to bf16 once; taps: 9, or 1 for a 1x1 window (padding
// 0, at kDown and kUp the even rows and columns).  The workspace may be null; one for the filter (Cout and Cin rounded up to 64
// by 18 bytes) makes large launches faster.  ADH_EUNIMPL: nothing launched, rows of fewer than two elements, or the launch is
// expected to take longer than `most_us`.
int conv_bf16_patch(const Conv3x3Problem &q, int taps, void *workspace, size_t workspace_bytes, double most_us, hipStream_t st);
// its kernel's name, or false where conv_bf16_patch takes nothing
bool conv_bf16_patch_name(const Conv3x3Problem &q, int taps, size_t workspace_bytes, double most_us, char *name, size_t name_bytes);

}  // namespace adh
#endif
