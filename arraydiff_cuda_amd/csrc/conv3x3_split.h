// The 3x3 window at stride 1, and at stride 2 over tiles without halo, in fp32, forward and backward-data: what conv3x3_split.hip gives the entry points.
#ifndef ADH_CONV3X3_SPLIT_H
#define ADH_CONV3X3_SPLIT_H

#include "adh_common.h"

namespace adh {

// out[m][R][Q] = beta*out + sum over c, a, b of w * in[c][R + D*a - pad_r][Q + D*b - pad_c], D the dilation (zero outside `in`)
// kDown, kUp: stride 2, padding 1, dilation 1 (tiles of even height and width), stacked without leading rows: forward from
// tiles of 2 step rows to such of step, and backward-data from the latter to the former
enum SplitSample { kUnit, kDown, kUp };
struct Conv3x3Problem {
  uint32_t num_tiles, N, C, M;  // C reduction channels, M produced channels
  // The tiles' extents.  stacked: they are the row tiles of one tensor in rank order, whose rows are numbered through: tile t
  // holds rows lead + t*step .. lead + (t+1)*step - 1 of it; `lead` rows precede the first tile's own and as many follow
  // the last one's (the padded forms' outer halo row).  Otherwise every tile is a tensor of its own.
  uint32_t in_H, in_W, out_H, out_W;
  SplitSample sample;
  bool stacked;
  uint32_t step, in_lead, out_lead;
  int32_t pad_r, pad_c;
  uint32_t dil;
  bool flip;  // backward-data: the filter is walked as w[c][m][8 - tap]
  float beta;
  const void *const *in, *const *res;  // res (may be null): what beta adds in place of the output
  void *const *out;
  const void *w;
  uint32_t w_m_stride, w_c_stride;  // of the filter's output and reduction channels
};

// The problem of the 3x3 entry points (conv3x3.hip).
Conv3x3Problem conv3x3_problem(int which, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W,
                               bool rows_from_neighbours, bool unpadded);

// fp32 sums of channel chunks that are dealt to several workgroups (0: none are)
size_t conv3x3_split_workspace(const Conv3x3Problem &q);
// The workspace may be null: then no chunks are dealt out.  ADH_EUNIMPL: nothing launched, as it is expected to take more than
// most_us, or as the shape is none that it takes.
int conv3x3_split(const Conv3x3Problem &q, void *workspace, size_t workspace_bytes, double most_us, hipStream_t st);
// whether it is expected to take more than most_us (or does not take the shape)
bool conv3x3_split_exceeds(const Conv3x3Problem &q, bool workspace, double most_us);
// more than one round of workgroups, and more than an eighth of all rounds idle
bool conv3x3_split_idles(const Conv3x3Problem &q);
void conv3x3_split_name(const Conv3x3Problem &q, char *name, size_t name_bytes);

}  // namespace adh
#endif
