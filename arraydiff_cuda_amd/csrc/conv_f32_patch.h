// Windows of 3x3 and 1x1 on fp32 tensors from patches in LDS, for launches that are too small for persistent workgroups: what
// conv_f32_patch.hip gives the entry points.
#ifndef ADH_CONV_F32_PATCH_H
#define ADH_CONV_F32_PATCH_H

#include "conv3x3_split.h"

namespace adh {

// taps: 9, or 1 for a 1x1 window (padding 0, at kDown and kUp the even rows and columns).
// Whether the 3x3 window is expected to be faster here than in conv3x3_split.hip (workspace: with one).
bool conv_f32_patch_ahead(const Conv3x3Problem &q, bool workspace);
// ADH_EUNIMPL: nothing launched, rows of fewer than two elements
int conv_f32_patch(const Conv3x3Problem &q, int taps, hipStream_t st);
bool conv_f32_patch_name(const Conv3x3Problem &q, int taps, char *name, size_t name_bytes);

}  // namespace adh
#endif
