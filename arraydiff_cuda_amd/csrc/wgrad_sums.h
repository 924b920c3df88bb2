// Filter gradients whose workgroups leave their sums in a workspace: the kernel that adds them.
//
// Workgroup (group, split) of a kernel with WO x WC waves owns 16*OT*WO output channels x 16*WC input channels x TAPS, each wave
// 16*OT x 16 as MFMA accumulators; its part is [wave][ot][tap][lane][4].  A group's parts follow each other, split by split.
#ifndef ADH_WGRAD_SUMS_H
#define ADH_WGRAD_SUMS_H

#include "split_bf16.h"

namespace adh {

struct WgradSums {
  float *part;  // [channel group][split][wave][ot][tap][lane][4]
  float *dw;    // [Cout][Cin][TAPS]
  uint32_t Cin, Cout, splits;
  float beta;
  FastDiv div_cig;  // channel group -> group of output channels, group of input channels
};

// dw = beta*dw + the splits' sums.  Sixteen lanes take sixteen neighbouring groups of four sums and 16 slices of the splits
// each (slice j: splits j, j + 16, ..); the slices are then added in order: a fixed order, so the result has fixed bits.  In
// double: as many fp32 additions of ever larger sums cost half a digit.
template <int TAPS, int OT, int WO, int WC>
__global__ __launch_bounds__(256) void wgrad_sums_kernel(const WgradSums P) {
  typedef double doublex4 __attribute__((ext_vector_type(4)));
  __shared__ doublex4 sums[16][16];
  constexpr uint32_t kQuads = WO * WC * OT * TAPS * 64u;  // of a channel group
  const uint32_t quad = blockIdx.x * 16u + (threadIdx.x & 15u), slice = threadIdx.x >> 4;
  const uint32_t group = quad / kQuads, e = quad - group * kQuads;
  const floatx4 *p = reinterpret_cast<const floatx4 *>(P.part) + (size_t)group * P.splits * kQuads + e;
  doublex4 sum = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4  // (eight, the compiler's choice: 16 -> 17 channels on 7 tiles of 24 x 440, 8 images, 46 us with the sums' kernel, 36 with four)
  for (uint32_t k = slice; k < P.splits; k += 16u) sum += __builtin_convertvector(*reinterpret_cast<const floatx4 *>(p + (size_t)k * kQuads), doublex4);
  sums[slice][threadIdx.x & 15u] = sum;
  __syncthreads();
  if (slice != 0u) return;
#pragma unroll
  for (int k = 1; k < 16; ++k) sum += sums[k][threadIdx.x];
  const uint32_t ln = e & 63u, rest = e >> 6, tap = rest % TAPS, ot = rest / TAPS % OT, wt = rest / TAPS / OT;
  uint32_t cog, cig;
  P.div_cig.divmod(group, cog, cig);
  const uint32_t co = cog * (16u * OT * WO) + ((wt % WO) * OT + ot) * 16u + (ln >> 4) * 4u, ci = cig * (16u * WC) + (wt / WO) * 16u + (ln & 15u);
  if (ci >= P.Cin) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (co + i >= P.Cout) break;
    float *d = P.dw + ((size_t)(co + i) * P.Cin + ci) * TAPS + tap;
    *d = (float)(P.beta != 0.f ? (double)*d + sum[i] : sum[i]);
  }
}

}  // namespace adh
#endif
