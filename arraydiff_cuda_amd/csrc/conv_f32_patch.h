// Windows of 3x3 and 1x1 on fp32 tensors from patches in LDS, for launches that are too small for persistent workgroups: what
// conv_f32_patch.hip gives the entry points.
#ifndef ADH_CONV_F32_PATCH_H
#define ADH_CONV_F32_PATCH_H

#include "conv_patch_plan.h"

namespace adh {

// taps: 9, or 1 for a 1x1 window (padding 0, at kDown and kUp the even rows and columns).
// The expected time of conv3x3_split.hip beyond which the 3x3 window is expected to be faster here, and the plan for that
// (1e300: it never is, and there is none).
double conv_f32_patch_beyond(const Conv3x3Problem &q, PatchPlan *plan);
int conv_f32_patch(const Conv3x3Problem &q, int taps, const PatchPlan &plan, hipStream_t st);
// ADH_EUNIMPL: nothing launched, rows of fewer than two elements
int conv_f32_patch(const Conv3x3Problem &q, int taps, hipStream_t st);
void conv_f32_patch_name(const Conv3x3Problem &q, int taps, const PatchPlan &plan, char *name, size_t name_bytes);

}  // namespace adh
#endif
