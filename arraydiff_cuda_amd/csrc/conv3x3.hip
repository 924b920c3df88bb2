// 3x3 convolution over the halo-padded slab and over row tiles without halo: the entry points, the arguments' checks, and
// the fp32 problem they describe (conv3x3_split.hip multiplies; bf16 tensors go to the kernels of conv3x3_bf16*.hip).
//   forward       : in = x, out = y,  Wt(o=co,k=ci,a,b) = w[co][ci][a][b]
//   backward-data : in = dy, out = dx, Wt(o=ci,k=co,a,b) = w[co][ci][2-a][2-b]; over padded tiles dx is the WHOLE padded slab
#include "conv3x3_split.h"
#include "conv_f32_patch.h"

#include <stdio.h>

namespace adh {

int conv_bf16_via_f32(int which, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W,
                      const void *const *in_tiles, const void *w, void *const *out_tiles, float beta, void *workspace,
                      size_t workspace_bytes, hipStream_t st);

// The problem of a pass whose tiles' interiors are H x W.  rows_from_neighbours: the tiles are the row tiles of one tensor
// in rank order; over padded tiles (forward) the inner halo rows are then the neighbours' interior rows, and (backward-data)
// what a halo reduce would add is part of the sums.  unpadded: neither side carries a halo.
Conv3x3Problem conv3x3_problem(int which, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W,
                               bool rows_from_neighbours, bool unpadded) {
  const bool fwd = which == ADH_CONV_FWD;
  const uint32_t halo = unpadded ? 0u : 2u;
  Conv3x3Problem q = {};
  q.num_tiles = num_tiles; q.N = N;
  q.C = fwd ? Cin : Cout; q.M = fwd ? Cout : Cin;
  q.in_H = H + (fwd ? halo : 0u); q.in_W = W + (fwd ? halo : 0u);
  q.out_H = H + (fwd ? 0u : halo); q.out_W = W + (fwd ? 0u : halo);
  q.stacked = rows_from_neighbours || unpadded;
  q.step = H;
  q.in_lead = fwd ? halo / 2u : 0u;
  q.out_lead = fwd ? 0u : halo / 2u;
  q.pad_r = q.pad_c = unpadded ? 1 : fwd ? 0 : 2;
  q.dil = 1;
  q.flip = !fwd;
  q.w_m_stride = fwd ? Cin * 9u : 9u;
  q.w_c_stride = fwd ? 9u : Cin * 9u;
  return q;
}

// which: ADH_CONV_FWD or ADH_CONV_BWD_DATA.  H, W are the interior extents.
static int conv_direct(int which, int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H,
                       uint32_t W, const void *const *in_tiles, const void *w, void *const *out_tiles, float beta,
                       hipStream_t st, bool rows_from_neighbours = false, bool unpadded = false,
                       const void *const *res_tiles = nullptr) {
  if (!dtype_ok(dtype)) return ADH_EINVAL;
  if (dtype != ADH_F32) return ADH_EUNIMPL;
  if (num_tiles == 0 || num_tiles > ADH_MAX_TILES) return ADH_EINVAL;
  if (beta != 0.f && beta != 1.f) return ADH_EINVAL;
  if (N == 0 || Cin == 0 || Cout == 0 || H == 0 || W == 0) return ADH_OK;
  if (!in_tiles || !out_tiles || !w) return ADH_ENULL;
  if (!aligned_to(w, 4)) return ADH_EALIGN;
  const uint64_t HP = (uint64_t)H + 2, WP = (uint64_t)W + 2;
  if (HP * WP >= (1ull << 31) || (uint64_t)N * num_tiles > 65535ull) return ADH_EINVAL;
  // one image and the filter are each addressed through a 32-bit buffer resource
  const uint64_t cmax = Cin > Cout ? Cin : Cout;
  if (cmax * HP * WP * 4u >= (1ull << 31) || (uint64_t)Cin * Cout * 36u >= (1ull << 31)) return ADH_EINVAL;
  for (uint32_t t = 0; t < num_tiles; ++t) {
    if (!in_tiles[t] || !out_tiles[t]) return ADH_ENULL;
    if (!aligned_to(in_tiles[t], 4) || !aligned_to(out_tiles[t], 4)) return ADH_EALIGN;
    if (res_tiles) {
      if (!res_tiles[t]) return ADH_ENULL;
      if (!aligned_to(res_tiles[t], 4)) return ADH_EALIGN;
    }
  }
  Conv3x3Problem q = conv3x3_problem(which, num_tiles, N, Cin, Cout, H, W, rows_from_neighbours, unpadded);
  q.beta = res_tiles ? 1.f : beta;
  q.in = in_tiles; q.out = out_tiles; q.res = res_tiles; q.w = w;
  // (of the plain form, for all forms of a layer: their sums have the same bits)
  PatchPlan patch = {};
  if (rows_from_neighbours) {
    const Conv3x3Problem plain = conv3x3_problem(which, num_tiles, N, Cin, Cout, H, W, false, unpadded);
    const double beyond = conv_f32_patch_beyond(plain, &patch);
    if (beyond == 1e300 || !conv3x3_split_exceeds(plain, false, beyond)) return conv3x3_split(q, nullptr, 0, 1e300, st);
    const int e = conv_f32_patch(q, 9, st);
    return e == ADH_EUNIMPL ? conv3x3_split(q, nullptr, 0, 1e300, st) : e;
  }
  const double beyond = conv_f32_patch_beyond(q, &patch);
  const int e = conv3x3_split(q, nullptr, 0, beyond, st);
  return e == ADH_EUNIMPL && beyond < 1e300 ? conv_f32_patch(q, 9, patch, st) : e;
}

// the patches' kernel name, where they serve the call
bool conv_bf16_takes_patches(int which, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W, char *name, size_t name_bytes);
const char *conv_bf16_kernel_name(int which, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W, float beta);
int conv_bf16_unpadded(int which, int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W,
                       const void *const *in_tiles, const void *w, void *const *out_tiles, float beta, void *workspace,
                       size_t workspace_bytes, hipStream_t st);

}  // namespace adh

using namespace adh;

extern "C" {

int adh_conv3x3_kernel_name(int which, int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout,
                            uint32_t H, uint32_t W, float beta, char *name, size_t name_bytes) {
  if (!name || name_bytes == 0) return ADH_ENULL;
  if (which != ADH_CONV_FWD && which != ADH_CONV_BWD_DATA) return ADH_EINVAL;
  if (num_tiles == 0 || N == 0 || Cin == 0 || Cout == 0 || H == 0 || W == 0) return ADH_EINVAL;
  if (dtype == ADH_BF16) {
    if (conv_bf16_takes_patches(which, num_tiles, N, Cin, Cout, H, W, name, name_bytes)) return ADH_OK;
    snprintf(name, name_bytes, "%s", conv_bf16_kernel_name(which, Cin, Cout, H, W, beta));
    return ADH_OK;
  }
  if (dtype != ADH_F32) return ADH_EINVAL;
  const Conv3x3Problem q = conv3x3_problem(which, num_tiles, N, Cin, Cout, H, W, false, false);
  PatchPlan patch = {};
  const double beyond = conv_f32_patch_beyond(q, &patch);
  if (beyond < 1e300 && conv3x3_split_exceeds(q, false, beyond)) conv_f32_patch_name(q, 9, patch, name, name_bytes);
  else conv3x3_split_name(q, name, name_bytes);
  return ADH_OK;
}

int adh_conv3x3_slab_fwd_tiles(int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H,
                               uint32_t W, const void *const *x_pad_tiles, const void *w, void *const *y_tiles,
                               float beta, void *workspace, size_t workspace_bytes, void *stream) {
  if (dtype == ADH_BF16)
    return conv_bf16_via_f32(ADH_CONV_FWD, num_tiles, N, Cin, Cout, H, W, x_pad_tiles, w, y_tiles, beta, workspace,
                             workspace_bytes, as_stream(stream));
  return conv_direct(ADH_CONV_FWD, dtype, num_tiles, N, Cin, Cout, H, W, x_pad_tiles, w, y_tiles, beta,
                     as_stream(stream));
}

int adh_conv3x3_slab_fwd_tiles_unexchanged(int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout,
                                           uint32_t H, uint32_t W, const void *const *x_pad_tiles, const void *w,
                                           void *const *y_tiles, float beta, void *workspace, size_t workspace_bytes,
                                           void *stream) {
  if (dtype == ADH_BF16) {
    // the bf16 kernels stream their rows from one image: exchange first, then the ordinary forward
    const int rc = adh_halo_exchange_nchw(dtype, 1, num_tiles, 1, W, H, Cin, N,
                                          const_cast<void *const *>(reinterpret_cast<const void *const *>(x_pad_tiles)),
                                          stream);
    if (rc != ADH_OK) return rc;
    return adh_conv3x3_slab_fwd_tiles(dtype, num_tiles, N, Cin, Cout, H, W, x_pad_tiles, w, y_tiles, beta, workspace,
                                      workspace_bytes, stream);
  }
  return conv_direct(ADH_CONV_FWD, dtype, num_tiles, N, Cin, Cout, H, W, x_pad_tiles, w, y_tiles, beta,
                     as_stream(stream), true);
}

int adh_conv3x3_slab_fwd(int dtype, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W,
                         const void *x_pad, const void *w, void *y, float beta, void *workspace,
                         size_t workspace_bytes, void *stream) {
  const void *xs[1] = {x_pad};
  void *ys[1] = {y};
  return adh_conv3x3_slab_fwd_tiles(dtype, 1, N, Cin, Cout, H, W, xs, w, ys, beta, workspace, workspace_bytes, stream);
}

int adh_conv3x3_slab_bwd_data_tiles(int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout,
                                    uint32_t H, uint32_t W, const void *w, const void *const *dy_tiles,
                                    void *const *dx_pad_tiles, float beta, void *workspace, size_t workspace_bytes,
                                    void *stream) {
  if (dtype == ADH_BF16)
    return conv_bf16_via_f32(ADH_CONV_BWD_DATA, num_tiles, N, Cin, Cout, H, W, dy_tiles, w, dx_pad_tiles, beta,
                             workspace, workspace_bytes, as_stream(stream));
  return conv_direct(ADH_CONV_BWD_DATA, dtype, num_tiles, N, Cin, Cout, H, W, dy_tiles, w, dx_pad_tiles, beta,
                     as_stream(stream));
}

int adh_conv3x3_slab_bwd_data_tiles_reduced(int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout,
                                            uint32_t H, uint32_t W, const void *w, const void *const *dy_tiles,
                                            void *const *dx_pad_tiles, float beta, void *workspace,
                                            size_t workspace_bytes, void *stream) {
  if (dtype == ADH_BF16) {
    // the bf16 kernels stream their rows from one image: the ordinary backward-data, then the reduce
    if (beta != 0.f) return ADH_EUNIMPL;  // a reduce after accumulating would add the old halo rows again
    const int rc = adh_conv3x3_slab_bwd_data_tiles(dtype, num_tiles, N, Cin, Cout, H, W, w, dy_tiles, dx_pad_tiles, beta,
                                                   workspace, workspace_bytes, stream);
    if (rc != ADH_OK) return rc;
    return adh_halo_reduce_nchw(dtype, 1, num_tiles, 1, W, H, Cin, N, dx_pad_tiles, stream);
  }
  return conv_direct(ADH_CONV_BWD_DATA, dtype, num_tiles, N, Cin, Cout, H, W, dy_tiles, w, dx_pad_tiles, beta,
                     as_stream(stream), true);
}

int adh_conv3x3_unpadded_fwd_tiles(int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H,
                                   uint32_t W, const void *const *x_tiles, const void *w, void *const *y_tiles, float beta,
                                   void *workspace, size_t workspace_bytes, void *stream) {
  if (dtype == ADH_F32)
    return conv_direct(ADH_CONV_FWD, dtype, num_tiles, N, Cin, Cout, H, W, x_tiles, w, y_tiles, beta, as_stream(stream),
                       true, true);
  return conv_bf16_unpadded(ADH_CONV_FWD, dtype, num_tiles, N, Cin, Cout, H, W, x_tiles, w, y_tiles, beta, workspace,
                            workspace_bytes, as_stream(stream));
}

int adh_conv3x3_unpadded_fwd_residual_tiles(int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H,
                                            uint32_t W, const void *const *x_tiles, const void *w,
                                            const void *const *res_tiles, void *const *y_tiles, void *stream) {
  if (!dtype_ok(dtype)) return ADH_EINVAL;
  if (dtype != ADH_F32) return ADH_EUNIMPL;
  if (!res_tiles) return ADH_ENULL;
  return conv_direct(ADH_CONV_FWD, dtype, num_tiles, N, Cin, Cout, H, W, x_tiles, w, y_tiles, 1.f, as_stream(stream), true,
                     true, res_tiles);
}

int adh_conv3x3_unpadded_bwd_data_tiles(int dtype, uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H,
                                        uint32_t W, const void *w, const void *const *dy_tiles, void *const *dx_tiles,
                                        float beta, void *workspace, size_t workspace_bytes, void *stream) {
  if (dtype == ADH_F32)
    return conv_direct(ADH_CONV_BWD_DATA, dtype, num_tiles, N, Cin, Cout, H, W, dy_tiles, w, dx_tiles, beta,
                       as_stream(stream), true, true);
  return conv_bf16_unpadded(ADH_CONV_BWD_DATA, dtype, num_tiles, N, Cin, Cout, H, W, dy_tiles, w, dx_tiles, beta, workspace,
                            workspace_bytes, as_stream(stream));
}

int adh_conv3x3_slab_bwd_data(int dtype, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W,
                              const void *w, const void *dy, void *dx_pad, float beta, void *workspace,
                              size_t workspace_bytes, void *stream) {
  const void *dys[1] = {dy};
  void *dxs[1] = {dx_pad};
  return adh_conv3x3_slab_bwd_data_tiles(dtype, 1, N, Cin, Cout, H, W, w, dys, dxs, beta, workspace, workspace_bytes,
                                         stream);
}

}  // extern "C"
