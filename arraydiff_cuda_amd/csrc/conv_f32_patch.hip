// 3x3 and 1x1 windows over fp32 tensors on the bf16 matrix cores (split_bf16.h says how), forward and backward-data, at stride 1 and 2,
// any width, any channel count, for launches that are too small for the persistent workgroups of conv3x3_split.hip:
//   out[m][R][Q] = beta*out + sum over c, a, b of w[m][c][a][b] * in[c][S*R + D*a - pad_r][S*Q + D*b - pad_c]
//
// Mapping: that of conv_bf16_patch.hip, in three parts.  A workgroup of four waves owns 16*MT output channels of 64*NT output pixels, a
// wave all of the channels and 16*NT of the pixels; per chunk of 32 channels (64 at 1x1) the patch and the chunk's filter, all
// taps of it, are split on their way to LDS as [part][octet of channels][pixel or channel][8 channels], and the next chunk is on
// its way to registers meanwhile: two barriers a chunk.  16 channels by 64 pixels take 77 KB, so that two workgroups share a
// compute unit; larger tiles have one to themselves.
//   * The products below h*h are summed apart from it, and the chunks' sums of it added as they come (few registers: the tiles are small):
//     relative error against double precision 0.9e-7 whatever the number of channels (in one chain 1.2e-7 from two chunks, 1.8e-7 from four).
//   * Sums that come out as NaN (an infinity's parts are not all finite) are computed over again in plain fp32.
// Measured (conv3x3_split.hip, at 1x1 the general kernel before), us, forward / backward-data: 480 -> 160 channels on 9 x 15 108 -> 38 /
// 40 -> 14; 44 -> 432, 2 images, 2 tiles of 12 x 29 forward 100 -> 33; 16 -> 224 on 2 tiles of 12 x 402 forward 56 -> 18; 115 layers of 16 to
// 512 channels 1.37 times as fast (geometric mean, including those that stay where they were).  Stride 2: 64 -> 128 channels, 6 images,
// 4 tiles of 28 x 40 backward-data 37 -> 17; forward 1.21, backward-data 1.44 in the mean of 45 blocks; 1x1 at stride 2 of 128 -> 128,
// 18 images of 42 x 78, forward 52 -> 16, 2 in the mean.
// Bound: by latency, a chunk's loads, splitting (half of the issued instructions), barriers and products one after the other.
#include "conv_f32_patch.h"

#include <stdio.h>

#include <algorithm>

#include "split_bf16.h"

namespace adh {

struct F32PatchParams : PatchParams {
  const void *res[ADH_MAX_TILES];  // what beta adds
};
typedef floatx2 pt_f32x2 __attribute__((aligned(4)));
typedef float pt_f32x3 __attribute__((ext_vector_type(3), aligned(4)));

// SAMPLE, TAPS: as in conv_bf16_patch.hip.
template <int MT, int NT, int SAMPLE, int TAPS>
__global__ __launch_bounds__(kPtThreads, 2) void conv_f32_patch_kernel(const F32PatchParams P) {
  constexpr uint32_t MW = 16u * MT, OCT = TAPS == 1 ? 8u : 4u, CHUNK = 8u * OCT;
  constexpr uint32_t PP = pt_pixels(SAMPLE, TAPS, NT, 3);
  constexpr bool SINGLE = SAMPLE == kDown && TAPS == 1;  // of a pair only the first pixel is of use
  constexpr int XU = (OCT * PP / (SINGLE ? 1u : 2u) + kPtThreads - 1u) / kPtThreads;  // (pair, octet) units a thread stages
  constexpr uint32_t GROUP = TAPS == 9 ? 3u : 1u, GROUPS = TAPS / GROUP;              // taps of a filter unit
  constexpr int WU = (MW * OCT * GROUPS + kPtThreads - 1u) / kPtThreads;              // (m, octet, group of taps) units
  constexpr int SETS = SAMPLE == kUp && TAPS == 9 ? 4 : 1;
  constexpr uint32_t DOWN = SAMPLE == kDown ? 2u : 1u, UP = SAMPLE == kUp ? 2u : 1u;
  constexpr uint32_t XP = OCT * PP, WP = TAPS * OCT * MW;  // of one part
  __shared__ __align__(16) uintx4 xl[3 * XP];
  __shared__ __align__(16) uintx4 wl[3 * WP];
  __shared__ const void *tab[3 * ADH_MAX_TILES];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));

  // neighbouring blocks (the channel groups of one block of pixels first) run on one XCD and share its cache
  const uint32_t vid = (blockIdx.x & 7u) * P.xcd_chunk + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= P.xcd_chunk || vid >= P.blocks) return;
  uint32_t outer, mg, group, inner, bi, bj;
  P.div_MG.divmod(vid, outer, mg);
  P.div_bpg.divmod(outer, group, inner);
  P.div_nbj.divmod(inner, bi, bj);
  const uint32_t img0 = group * P.NB;

  // (a per-lane choice of tile would be looked up one lane group at a time from the kernel's arguments)
  if (tid < P.num_tiles) {
    tab[tid] = P.in[tid];
    tab[ADH_MAX_TILES + tid] = P.out[tid];
    tab[2 * ADH_MAX_TILES + tid] = P.res[tid];
  }
  lds_barrier();
  auto in_tile = [&](uint32_t R) { return R < P.in_lead ? 0u : min(P.div_in.div(R - P.in_lead), P.last_tile); };
  auto out_tile = [&](uint32_t R) { return R < P.out_lead ? 0u : min(P.div_out.div(R - P.out_lead), P.last_tile); };

  // ---- the patch: this thread stages units tid + j * 256 of its pairs' octets (octet 0 of all pairs first) ----
  const size_t plane = (size_t)P.in_H * P.in_W;
  const ADH_GLOBAL char *xp[XU];  // the pair in the first channel of the unit's octet of the next chunk
  uint32_t xsel[XU], xat[XU];     // which of the pair its pixels are (0: none, 1, 2; the second pixel's times 4); where they go
  floatx2 xv[XU][8];
#pragma unroll
  for (int j = 0; j < XU; ++j) {
    uint32_t o, p, b, e, r, k;
    P.div_pairs.divmod(tid + (uint32_t)j * kPtThreads, o, p);
    P.div_pairs_img.divmod(p, b, e);
    P.div_pairs_row.divmod(e, r, k);
    const uint32_t img = img0 + b;
    const int32_t R = (int32_t)((bi * P.BR + (SINGLE ? r : 0u)) * DOWN + (SINGLE ? 0u : r)) - P.pad_r, Q = (int32_t)(bj * P.BC * DOWN + 2u * k) - P.pad_c;
    const bool live = o < OCT && 8u * o < P.C && img < P.NI && R >= 0 && R < (int32_t)P.in_VH;
    uint32_t tile0, n;
    P.div_N.divmod(live ? img : 0u, tile0, n);
    const uint32_t Ru = live ? (uint32_t)R : P.in_lead, t = in_tile(Ru);
    const int32_t Qc = min(max(Q, 0), (int32_t)P.in_W - 2), s = Q - Qc;  // the existing pair at Qc holds pixel Q at s, Q + 1 at s + 1
    xsel[j] = !live ? 0u : (s == 0 ? 1u : s == 1 ? 2u : 0u) | (s == -1 ? 4u : s == 0 ? 8u : 0u);
    xat[j] = o * PP + b * P.image + r * P.pitch + (SAMPLE == kDown ? k : 2u * k);
    xat[j] = o < OCT ? xat[j] : ~0u;
    // (a unit that does not exist loads an existing place; its values are replaced by zero)
    xp[j] = (const ADH_GLOBAL char *)tab[tile0 + t] +
            (((size_t)n * P.C + (live ? 8u * o : 0u)) * plane + (size_t)(Ru - t * P.in_step) * P.in_W + (uint32_t)Qc) * 4u;
  }
  const size_t step = plane * 4u;
  auto load_x = [&](uint32_t ch) {
    const bool whole = (ch + 1u) * CHUNK <= P.C;
#pragma unroll
    for (int j = 0; j < XU; ++j) {
      if (wave * 64u + (uint32_t)j * kPtThreads >= OCT * P.div_pairs.d) break;
      const ADH_GLOBAL char *p = xp[j];
      if (whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          xv[j][e] = *(const ADH_GLOBAL pt_f32x2 *)p;
          p += step;
        }
      } else {
        // past the last channel the address stays, and an octet without any keeps the one it loaded last
        const uint32_t c0 = ch * CHUNK + P.div_pairs.div(tid + (uint32_t)j * kPtThreads) * 8u;
        if (c0 >= P.C) p -= ch ? CHUNK * step : (size_t)0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          xv[j][e] = *(const ADH_GLOBAL pt_f32x2 *)p;
          if (c0 + e + 1u < P.C) p += step;
        }
      }
      xp[j] += CHUNK * step;
    }
  };
  auto store_x = [&](uint32_t ch) {
    const bool whole = (ch + 1u) * CHUNK <= P.C;
#pragma unroll
    for (int j = 0; j < XU; ++j) {
      if (wave * 64u + (uint32_t)j * kPtThreads >= OCT * P.div_pairs.d) break;
      if (!whole) {
        const uint32_t c0 = ch * CHUNK + P.div_pairs.div(tid + (uint32_t)j * kPtThreads) * 8u;
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[j][e] = c0 + e < P.C ? xv[j][e] : floatx2{0.f, 0.f};
      }
      if (xsel[j] != 9u) {
        const uint32_t a = xsel[j] & 3u, b = xsel[j] >> 2;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const floatx2 v = xv[j][e];
          xv[j][e] = floatx2{a == 1u ? v[0] : a == 2u ? v[1] : 0.f, b == 1u ? v[0] : b == 2u ? v[1] : 0.f};
        }
      }
#pragma unroll
      for (int h = 0; h < (SINGLE ? 1 : 2); ++h) {
        uint32_t part[3][4];
#pragma unroll
        for (int d = 0; d < 4; ++d) split_pair(xv[j][2 * d][h], xv[j][2 * d + 1][h], part[0][d], part[1][d], part[2][d]);
        if (xat[j] != ~0u) {
#pragma unroll
          for (int k = 0; k < 3; ++k)
            xl[k * XP + xat[j] + (h ? (SAMPLE == kDown ? P.BC + 1u : 1u) : 0u)] = uintx4{part[k][0], part[k][1], part[k][2], part[k][3]};
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- the filter: eight channels' GROUP neighbouring taps of an output channel a unit ----
  float wv[WU][8][GROUP];
  struct FilterUnit { uint32_t m, o, t; };
  auto w_unit = [&](int j) {  // forward, lanes run over taps and octets first: what they want then lies side by side
    const uint32_t u = tid + (uint32_t)j * kPtThreads, r = u / GROUPS, t = u % GROUPS;
    return P.flip ? FilterUnit{r % MW, r / MW, t} : FilterUnit{r / OCT, r % OCT, t};
  };
  auto load_w = [&](uint32_t ch) {
#pragma unroll
    for (int j = 0; j < WU; ++j) {
      if (wave * 64u + (uint32_t)j * kPtThreads >= MW * OCT * GROUPS) break;
      const FilterUnit F = w_unit(j);
      const uint32_t c0 = ch * CHUNK + 8u * F.o;
      const ADH_GLOBAL float *p = (const ADH_GLOBAL float *)P.w + (size_t)min(mg * MW + F.m, P.M - 1u) * P.w_m_stride + (size_t)min(c0, P.C - 1u) * P.w_c_stride + F.t * GROUP;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (GROUP == 3u) {
          const pt_f32x3 v = *(const ADH_GLOBAL pt_f32x3 *)p;
          wv[j][e][0] = v[0]; wv[j][e][1] = v[1]; wv[j][e][2] = v[2];
        } else {
          wv[j][e][0] = *p;
        }
        p += c0 + e + 1u < P.C ? P.w_c_stride : 0u;
      }
    }
  };
  auto store_w = [&](uint32_t ch) {
#pragma unroll
    for (int j = 0; j < WU; ++j) {
      if (wave * 64u + (uint32_t)j * kPtThreads >= MW * OCT * GROUPS) break;
      const FilterUnit F = w_unit(j);
      if ((ch + 1u) * CHUNK > P.C) {  // (channels that do not exist multiply zeros: an infinity must not)
        const uint32_t c0 = ch * CHUNK + 8u * F.o;
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (uint32_t i = 0; i < GROUP; ++i) wv[j][e][i] = c0 + e < P.C ? wv[j][e][i] : 0.f;
      }
#pragma unroll
      for (uint32_t i = 0; i < GROUP; ++i) {
        uint32_t part[3][4];
#pragma unroll
        for (int d = 0; d < 4; ++d) split_pair(wv[j][2 * d][i], wv[j][2 * d + 1][i], part[0][d], part[1][d], part[2][d]);
        const uint32_t t = F.t * GROUP + i;
#pragma unroll
        for (int k = 0; k < 3; ++k) wl[k * WP + ((P.flip ? TAPS - 1u - t : t) * OCT + F.o) * MW + F.m] = uintx4{part[k][0], part[k][1], part[k][2], part[k][3]};
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- this wave's pixels: 16 consecutive ones of the block's NB x BR x BC per tile ----
  uint32_t pix[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    uint32_t b, e, r, c;
    P.div_live.divmod((wave * NT + q) * 16u + l16, b, e);
    P.div_BC.divmod(e, r, c);
    pix[q] = (b < P.NB ? b * P.image + r * (SINGLE ? 1u : DOWN) * P.pitch + c : 0u) + g * PP;
  }
  auto tap_place = [&](uint32_t a, uint32_t b) {
    if constexpr (TAPS == 1) return 0u;
    else if constexpr (SAMPLE == kDown) return a * P.pitch + (b == 1u ? P.BC + 1u : b / 2u);
    else if constexpr (SAMPLE == kUp) return a / 2u * P.pitch + b / 2u;
    else return (a * P.pitch + b) * P.dil;
  };
  auto tap_set = [](int t) { return SETS == 4 ? (t / 3 == 1 ? 0 : 2) + (t % 3 == 1 ? 0 : 1) : 0; };
  floatx4 acc[SETS][MT][NT], low[SETS][MT][NT], sums[SETS][MT][NT];  // a chunk's h*h, the small products apart, the chunks' sums
#pragma unroll
  for (int s = 0; s < SETS; ++s)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < NT; ++q) sums[s][mt][q] = low[s][mt][q] = floatx4{0.f, 0.f, 0.f, 0.f};
  const uintx4 *const f_lane = wl + g * MW + l16;

  load_w(0);
  load_x(0);
  for (uint32_t ch = 0; ch < P.nchunks; ++ch) {
    if (ch) lds_barrier();
    store_w(ch);
    store_x(ch);
    lds_barrier();
    if (ch + 1u < P.nchunks) {
      load_w(ch + 1u);
      load_x(ch + 1u);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int q = 0; q < NT; ++q) acc[s][mt][q] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < TAPS; ++t) {
      const uint32_t delta = tap_place(t / 3, t % 3);
#pragma unroll
      for (uint32_t ks = 0; ks < OCT / 4u; ++ks) {
        uintx4 x[NT][3], f[MT][3];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int k = 0; k < 3; ++k) f[mt][k] = f_lane[k * WP + (t * OCT + ks * 4u) * MW + mt * 16];
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
          for (int k = 0; k < 3; ++k) x[q][k] = xl[k * XP + pix[q] + delta + ks * 4u * PP];
        auto products = [&](floatx4 (&sum)[MT][NT], int kx, int kf) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int q = 0; q < NT; ++q) sum[mt][q] = mfma_bf16(x[q][kx], f[mt][kf], sum[mt][q]);
        };
        auto &lo = low[tap_set(t)];
        products(lo, 0, 2); products(lo, 1, 1); products(lo, 2, 0); products(lo, 0, 1); products(lo, 1, 0);
        products(acc[tap_set(t)], 0, 0);
      }
    }
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int q = 0; q < NT; ++q) sums[s][mt][q] += acc[s][mt][q];
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- results: a lane has four neighbouring pixels of a row (block widths are multiples of four) of channel 16 mt + l16 ----
  const size_t out_plane = (size_t)P.out_H * P.out_W;
  const uint32_t m0 = mg * MW + l16;
  // result (m, R, Q) of an image once more in plain fp32
  auto plain = [&](uint32_t tile0, uint32_t n, uint32_t m, uint32_t R, uint32_t Q) {
    float sum = 0.f;
    for (uint32_t t = 0; t < (uint32_t)TAPS; ++t) {
      const uint32_t a = t / 3u, b = t % 3u;
      int32_t r, q;
      if (SAMPLE == kUp) {
        if (TAPS == 9 ? ((R & 1u) != 0u) != (a != 1u) || ((Q & 1u) != 0u) != (b != 1u) : ((R | Q) & 1u) != 0u) continue;
        r = (int32_t)(R / 2u + (TAPS == 9 ? a / 2u : 0u));
        q = (int32_t)(Q / 2u + (TAPS == 9 ? b / 2u : 0u));
      } else {
        r = (int32_t)(R * DOWN + a * (SAMPLE == kUnit ? P.dil : 1u)) - P.pad_r;
        q = (int32_t)(Q * DOWN + b * (SAMPLE == kUnit ? P.dil : 1u)) - P.pad_c;
      }
      const bool exists = r >= 0 && r < (int32_t)P.in_VH && q >= 0 && q < (int32_t)P.in_W;  // (the padding is data: an infinite filter element times it is NaN)
      const uint32_t it = exists ? in_tile((uint32_t)r) : 0u;
      const ADH_GLOBAL float *in = (const ADH_GLOBAL float *)tab[tile0 + it] + (size_t)n * P.C * plane + (exists ? (size_t)((uint32_t)r - it * P.in_step) * P.in_W + (uint32_t)q : (size_t)0);
      const ADH_GLOBAL float *f = (const ADH_GLOBAL float *)P.w + (size_t)m * P.w_m_stride + (P.flip ? TAPS - 1u - t : t);
      for (uint32_t c = 0; c < P.C && sum == sum; ++c) sum = __builtin_fmaf(exists ? in[(size_t)c * plane] : 0.f, f[(size_t)c * P.w_c_stride], sum);
    }
    return sum;
  };
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    uint32_t b, e, r, c, tile0, n;
    P.div_live.divmod((wave * NT + q) * 16u + 4u * g, b, e);
    P.div_BC.divmod(e, r, c);
    const uint32_t img = img0 + b, i = bi * P.BR + r, j = bj * P.BC + c;
    if (b >= P.NB || img >= P.NI || i >= P.grid_VH || j >= P.grid_W) continue;
    P.div_N.divmod(img, tile0, n);
    const uint32_t t = out_tile(i);
    const size_t at0 = ((size_t)n * P.M + m0) * out_plane + (size_t)((i - t * P.out_step) * UP) * P.out_W + j * UP;
    ADH_GLOBAL float *const out = (ADH_GLOBAL float *)tab[ADH_MAX_TILES + tile0 + t] + at0;
    const ADH_GLOBAL float *const res = (const ADH_GLOBAL float *)tab[2 * ADH_MAX_TILES + tile0 + t] + at0;
    const uint32_t count = min(4u, P.grid_W - j);  // (quads) of this lane that exist
    // 4 N results side by side from `at` on, some of them existing; of output row R, column Q on
    auto emit = [&](size_t at, auto &v, uint32_t exist, uint32_t m, uint32_t R, uint32_t Q) {
      constexpr int N = sizeof(v) / sizeof(floatx4);
      bool nan = false;
#pragma unroll
      for (int h = 0; h < N; ++h) nan |= __builtin_isunordered(v[h][0], v[h][1]) || __builtin_isunordered(v[h][2], v[h][3]);
      if (nan) {
#pragma unroll
        for (int k = 0; k < 4 * N; ++k)
          if ((uint32_t)k < exist && v[k / 4][k % 4] != v[k / 4][k % 4]) v[k / 4][k % 4] = plain(tile0, n, m, R, Q + k);
      }
#pragma unroll
      for (int h = 0; h < N; ++h) {
        if (exist >= 4u * h + 4u) {
          if (P.beta != 0.f) v[h] += *(const ADH_GLOBAL floatx4_u *)(res + at + 4 * h);
          *(ADH_GLOBAL floatx4_u *)(out + at + 4 * h) = v[h];
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (4u * h + k < exist) out[at + 4 * h + k] = v[h][k] + (P.beta != 0.f ? res[at + 4 * h + k] : 0.f);
        }
      }
    };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const uint32_t m = m0 + mt * 16u;
      if (m >= P.M) break;
      const size_t at = (size_t)(mt * 16) * out_plane;
      floatx4 v[SETS];
#pragma unroll
      for (int s = 0; s < SETS; ++s) v[s] = sums[s][mt][q] + low[s][mt][q];
      if constexpr (SAMPLE == kUp) {
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          floatx4 w[2];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            w[k / 2][2 * (k % 2)] = SETS == 4 ? v[SETS == 4 ? 2 * pr : 0][k] : pr ? 0.f : v[0][k];
            w[k / 2][2 * (k % 2) + 1] = SETS == 4 ? v[SETS == 4 ? 2 * pr + 1 : 0][k] : 0.f;
          }
          emit(at + (pr ? P.out_W : 0u), w, 2u * count, m, 2u * i + pr, 2u * j);
        }
      } else {
        floatx4 w[1] = {v[0]};
        emit(at, w, count, m, i, j);
      }
    }
  }
}

// ---- host side ----

template <int MT, int SAMPLE, int TAPS>
static void launch_f32_patch(const PatchPlan &plan, const F32PatchParams &P, hipStream_t st) {
  const dim3 grid(P.xcd_chunk * 8u), block(kPtThreads);
  if constexpr (SAMPLE == kUnit || TAPS == 1) {
    if (plan.NT == 2) {
      hipLaunchKernelGGL((conv_f32_patch_kernel<MT, 2, SAMPLE, TAPS>), grid, block, 0, st, P);
      return;
    }
  }
  hipLaunchKernelGGL((conv_f32_patch_kernel<MT, 1, SAMPLE, TAPS>), grid, block, 0, st, P);
}
template <int SAMPLE, int TAPS>
static void launch_f32_patch_mt(const PatchPlan &plan, const F32PatchParams &P, hipStream_t st) {
  plan.MT == 2 ? launch_f32_patch<2, SAMPLE, TAPS>(plan, P, st) : launch_f32_patch<1, SAMPLE, TAPS>(plan, P, st);
}

// The expected times of both are fitted to 230 launches at stride 1 and 90 at stride 2 (rms error 5 - 8 % here, 11 - 15 % there); at
// stride 1 patches have to be expected 5 % ahead: of 2241 passes of random layers 10 lose more than 3 % by them, up to 17 % (22 and 24 %
// without), 0.4 % more time over all than with the better of both each time.  Patches are ahead up to some 30 us,
// 3 times at the smallest, where the other kernel's nine barriers a chunk and its filter tap by tap stand in a row (480 -> 160
// channels on 9 x 15, forward 108 -> 38 us); persistent workgroups of twice the waves where blocks are many.
// (Beyond four rounds of the smallest blocks they are 0.5 to 1.1 times as fast and not priced: the choice is made on every call.)
// Host time: planned once a call and the other kernel not where its least time says enough: 16 -> 16 channels on 2 tiles of 4 x 2000 2.7 -> 0.5 us.
double conv_f32_patch_beyond(const Conv3x3Problem &q, PatchPlan *plan) {
  const uint64_t pixels = (uint64_t)q.num_tiles * q.N * (q.sample == kUp ? (uint64_t)q.in_H * q.in_W : (uint64_t)q.out_H * q.out_W);
  if (pixels * q.M > 2048ull * 64u * 16u || patch_plan(q, 9, 3, 0u, plan)) return 1e300;
  if (q.sample == kDown) return (1.2 * plan->us - 3.3) / 1.23;
  if (q.sample == kUp) return (1.13 * plan->us - 0.7) / 1.1;  // (1.07 as fitted; 512 -> 512 channels on 4 x 16 tiles lost 4 % by it)
  return (1.05 * plan->us - 3.5) / 1.09;
}

void conv_f32_patch_name(const Conv3x3Problem &q, int taps, const PatchPlan &plan, char *name, size_t name_bytes) {
  snprintf(name, name_bytes, "conv_f32_patch_kernel<%d, %d, %d, %d>", plan.MT, plan.NT, (int)q.sample, taps);
}

int conv_f32_patch(const Conv3x3Problem &q, int taps, hipStream_t st) {
  PatchPlan plan = {};
  const int e = patch_plan(q, taps, 3, 0u, &plan);
  return e ? e : conv_f32_patch(q, taps, plan, st);
}

int conv_f32_patch(const Conv3x3Problem &q, int taps, const PatchPlan &plan, hipStream_t st) {
  F32PatchParams P = {};
  static_cast<PatchParams &>(P) = plan.P;
  for (uint32_t t = 0; t < q.num_tiles; ++t) {
    P.in[t] = q.in[t];
    P.out[t] = q.out[t];
    P.res[t] = q.res ? q.res[t] : q.out[t];
  }
  P.w = q.w;
  if (taps == 9) {
    if (q.sample == kUnit) launch_f32_patch_mt<kUnit, 9>(plan, P, st);
    else if (q.sample == kDown) launch_f32_patch_mt<kDown, 9>(plan, P, st);
    else launch_f32_patch_mt<kUp, 9>(plan, P, st);
  } else {
    if (q.sample == kUnit) launch_f32_patch_mt<kUnit, 1>(plan, P, st);
    else if (q.sample == kDown) launch_f32_patch_mt<kDown, 1>(plan, P, st);
    else launch_f32_patch_mt<kUp, 1>(plan, P, st);
  }
  return launch_status();
}

}  // namespace adh
