// How windows on patches in LDS are cut into blocks: conv_bf16_patch.hip, conv_f32_patch.hip.
#ifndef ADH_CONV_PATCH_PLAN_H
#define ADH_CONV_PATCH_PLAN_H

#include "conv3x3_split.h"

namespace adh {

constexpr uint32_t kPtThreads = 256;
// pixels of a patch plane in LDS (parts: 1, bf16; 3, fp32 in three parts)
constexpr uint32_t pt_pixels(int sample, int taps, int nt, int parts) {
  if (parts == 3 && taps == 9 && sample == kDown) return 320u;
  return taps == 1 ? 64u * nt + 16u : sample == kDown ? 640u : nt == 4 ? 640u : nt == 2 ? 384u : 256u;
}

struct PatchParams {
  const void *in[ADH_MAX_TILES];
  void *out[ADH_MAX_TILES];
  const void *w;  // the caller's, or (READY) in the order of the LDS: [64 m][chunk][tap][octet][m][8 channels]
  uint32_t N, NI, C, M, num_tiles;
  uint32_t in_H, in_W, out_H, out_W;
  uint32_t in_VH, grid_VH, grid_W;  // rows of the (stacked) input; what the blocks tile: output pixels, or quads of them
  uint32_t in_lead, out_lead, in_step, out_step, last_tile;
  uint32_t w_m_stride, w_c_stride;
  uint32_t BR, BC, NB, pitch, image;  // a block's pixels: BR x BC of NB images; pixels of a patch row, of an image's patch
  uint32_t nchunks, blocks, xcd_chunk;
  int32_t pad_r, pad_c, flip;
  uint32_t dil;
  float beta;
  FastDiv div_bpg, div_nbj, div_MG, div_N, div_BC, div_live, div_pairs, div_pairs_img, div_pairs_row, div_in, div_out;
};

struct PatchPlan {
  PatchParams P;
  int MT, NT;
  bool ready;    // the filter is put in order first
  uint64_t units;  // of eight channels' taps in it
  double us;     // what the launches are expected to take
};

int patch_plan(const Conv3x3Problem &q, int taps, int parts, size_t workspace_bytes, PatchPlan *plan);

}  // namespace adh
#endif
