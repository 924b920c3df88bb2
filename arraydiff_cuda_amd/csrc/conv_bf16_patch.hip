// 3x3 and 1x1 windows over bf16 tensors on the matrix cores, forward and backward-data, at stride 1 and 2, any width, any
// channel count, all reduction channels in one launch:
//   out[m][R][Q] = beta*out + sum over c, a, b of w[m][c][a][b] * in[c][S*R + D*a - pad_r][S*Q + D*b - pad_c]
//
// Mapping.  v_mfma_f32_16x16x32_bf16, k = 32 channels of one tap.  A workgroup of four waves, two per compute unit, owns 16*MT
// output channels of 64*NT output pixels; a wave all of the channels and 16*NT of the pixels.
//   * The input patch of a chunk of channels lies in LDS as [octet of channels][pixel][8 channels]: an operand is one
//     ds_read_b128 of neighbouring pixels whatever the tap.  A thread loads two neighbouring pixels of a row (4 bytes at any
//     alignment) from eight channels' planes and puts them in order with byte permutes, whose selectors also make the zeros
//     of the padding: no lane asks memory for more than an existing pair.
//   * The filter is read as the caller holds it (nine elements of a channel side by side) and reordered the same way.
//   * The next chunk is on its way to registers while this one is multiplied.  One LDS buffer: the other workgroup of the
//     compute unit multiplies meanwhile.
// Measured (general kernels, which widen to fp32 -> here).  3x3 at stride 2, 128 -> 256 channels, 32 images, 4 tiles of 16 x 64: forward
// and backward-data with the 1x1 of the same stride 840 -> 180 us (65 / 48 / 19 / 48); 56 -> 112, 2 images, 2 tiles of 22 x 124: 115 -> 36.
// At stride 1 the choice between strips and patches (conv3x3_bf16_mfma.hip) holds both sides.
// Bound: large launches by latency (matrix pipes busy 0.2 to 0.45 of the time; a block of one or two chunks waits for its first
// patch) and by LDS, whose reads at MT = NT = 4 take as long as the multiplications.  Padding the operands' planes in LDS costs 2
// to 7 %, half the tile (no spilled registers) 4 to 40 %.
#include "conv_bf16_patch.h"

#include "conv_patch_plan.h"

#include <stdio.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "split_bf16.h"

namespace adh {

typedef uint32_t pt_u32 __attribute__((aligned(2)));
typedef uintx4 pt_u32x4 __attribute__((aligned(2)));
typedef uintx2 pt_u32x2 __attribute__((aligned(2)));

constexpr uint32_t kPickLow = 0x05040100u, kPickHigh = 0x07060302u, kPickZero = 0x0c0c0c0cu;
// low (high) halves of a and b side by side, a's below
__device__ __forceinline__ uint32_t pt_pick(uint32_t a, uint32_t b, uint32_t sel) { return __builtin_amdgcn_perm(b, a, sel); }
__device__ __forceinline__ uint32_t pt_round(float a, float b) {
  const floatx2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// N channels from c0 on of one output channel's filter: TAPS elements side by side each, `stride` elements apart (past the
// last channel an existing one).
template <int TAPS, int N, int WR>
__device__ __forceinline__ void pt_load_filter(const uint16_t *p, uint32_t c0, uint32_t C, uint32_t stride, uint32_t (&v)[N][WR]) {
#pragma unroll
  for (int e = 0; e < N; ++e) {
    if constexpr (TAPS == 9) {
      const uintx4 a = *(const ADH_GLOBAL pt_u32x4 *)p;
      v[e][0] = a[0]; v[e][1] = a[1]; v[e][2] = a[2]; v[e][3] = a[3];
      v[e][4] = *(const ADH_GLOBAL uint16_t *)(p + 8);
    } else {
      v[e][0] = *(const ADH_GLOBAL uint16_t *)p;
    }
    p += c0 + e + 1u < C ? stride : 0u;
  }
}
// (channels that do not exist multiply zeros: an infinity must not)
template <int N, int WR>
__device__ __forceinline__ void pt_mask_filter(uint32_t c0, uint32_t C, uint32_t (&v)[N][WR]) {
#pragma unroll
  for (int e = 0; e < N; ++e)
#pragma unroll
    for (int r = 0; r < WR; ++r) v[e][r] = c0 + e < C ? v[e][r] : 0u;
}
template <int N, int WR>
__device__ __forceinline__ auto pt_filter_tap(int t, const uint32_t (&v)[N][WR]) {
  uint32_t r[N / 2];
#pragma unroll
  for (int d = 0; d < N / 2; ++d) r[d] = pt_pick(v[2 * d][t / 2], v[2 * d + 1][t / 2], t % 2 ? kPickHigh : kPickLow);
  if constexpr (N == 8) return uintx4{r[0], r[1], r[2], r[3]};
  else if constexpr (N == 4) return uintx2{r[0], r[1]};
  else return r[0];
}

// The caller's filter in the order of the LDS: a thread per (64 m, chunk, octet, m).
__global__ __launch_bounds__(kPtThreads) void conv_bf16_patch_filter_kernel(const uint16_t *w, uintx4 *ready, uint32_t M, uint32_t C,
                                                                            uint32_t nchunks, uint32_t m_stride, uint32_t c_stride, int flip, uint32_t units) {
  const uint32_t u = blockIdx.x * kPtThreads + threadIdx.x;
  if (u >= units) return;
  const uint32_t m64 = u % 64u, o = u / 64u % 4u, block = u / 256u, ch = block % nchunks, m = block / nchunks * 64u + m64, c0 = ch * 32u + 8u * o;
  uint32_t v[8][5];
  pt_load_filter<9>(w + (size_t)min(m, M - 1u) * m_stride + (size_t)min(c0, C - 1u) * c_stride, c0, C, c_stride, v);
  pt_mask_filter(c0, C, v);
#pragma unroll
  for (int t = 0; t < 9; ++t) ready[((size_t)block * 9u + (flip ? 8 - t : t)) * 256u + o * 64u + m64] = pt_filter_tap(t, v);
}

// SAMPLE.  kDown (stride 2): the patch holds a row's first, third, .. columns, then the others, so that the 16 pixels of an
// operand are neighbours in LDS for every tap.  kUp (backward-data at stride 2): a block owns quads, the 2 x 2 gradient pixels at
// (2i, 2j), which tap (1 +- a, 1 +- b) of the filter feeds from dy[i .. i + 1][j .. j + 1], into four sets of sums.
template <int MT, int NT, int SAMPLE, int TAPS, bool READY>
__global__ __launch_bounds__(kPtThreads, 2) void conv_bf16_patch_kernel(const PatchParams P) {
  constexpr uint32_t MW = 16u * MT, OCT = TAPS == 1 ? 8u : 4u, CHUNK = 8u * OCT;
  constexpr uint32_t PP = pt_pixels(SAMPLE, TAPS, NT, 1);
  constexpr bool SINGLE = SAMPLE == kDown && TAPS == 1;  // of a pair only the first pixel is of use
  constexpr int XU = (OCT * PP / (SINGLE ? 1u : 2u) + kPtThreads - 1u) / kPtThreads;  // (pair, octet) units a thread stages
  // filter units: WC of an octet's channels.  Small tiles' are cut so that all threads have as many (one wave's 64 octets of 16 output
  // channels kept the others waiting: forward 1.07 to 1.11, backward-data 1.02 to 1.04 times as fast without; at larger tiles 0.97 to 1.05).
  constexpr uint32_t WC = MT * NT <= 2 && MW * OCT / 32u < 8u ? MW * OCT / 32u : 8u, SUB = 8u / WC;
  constexpr uint32_t WUNITS = MW * OCT * SUB;
  constexpr int WU = (int)((WUNITS + kPtThreads - 1u) / kPtThreads);
  constexpr int WR = TAPS == 9 ? 5 : 1;
  constexpr int SETS = SAMPLE == kUp && TAPS == 9 ? 4 : 1;
  constexpr uint32_t DOWN = SAMPLE == kDown ? 2u : 1u, UP = SAMPLE == kUp ? 2u : 1u;
  __shared__ __align__(16) uintx4 xl[OCT * PP];
  __shared__ __align__(16) uintx4 wl[TAPS * OCT * MW];
  __shared__ const void *tab[2 * ADH_MAX_TILES];
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
  }
  lds_barrier();
  auto in_tile = [&](uint32_t R) { return R < P.in_lead ? 0u : min(P.div_in.div(R - P.in_lead), P.last_tile); };
  auto out_tile = [&](uint32_t R) { return R < P.out_lead ? 0u : min(P.div_out.div(R - P.out_lead), P.last_tile); };

  // ---- the patch: this thread stages units tid + j * 256 of its pairs' octets (octet 0 of all pairs first) ----
  const size_t plane = (size_t)P.in_H * P.in_W;
  const ADH_GLOBAL char *xp[XU];   // the pair in the first channel of the unit's octet of the next chunk
  uint32_t xsel[XU][2], xat[XU];   // how its pixels are picked; where they go
  uint32_t xv[XU][8];
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
    xsel[j][0] = !live || s < 0 || s > 1 ? kPickZero : s == 0 ? kPickLow : kPickHigh;
    xsel[j][1] = !live || s < -1 || s > 0 ? kPickZero : s == 0 ? kPickHigh : kPickLow;
    xat[j] = o * PP + b * P.image + r * P.pitch + (SAMPLE == kDown ? k : 2u * k);
    xat[j] = o < OCT ? xat[j] : ~0u;
    // (a unit that does not exist loads an existing place; its values are replaced by zero)
    xp[j] = (const ADH_GLOBAL char *)tab[tile0 + t] +
            (((size_t)n * P.C + (live ? 8u * o : 0u)) * plane + (size_t)(Ru - t * P.in_step) * P.in_W + (uint32_t)Qc) * 2u;
  }
  const size_t step = plane * 2u;
  auto load_x = [&](uint32_t ch) {
    const bool whole = (ch + 1u) * CHUNK <= P.C;
#pragma unroll
    for (int j = 0; j < XU; ++j) {
      if (wave * 64u + (uint32_t)j * kPtThreads >= OCT * P.div_pairs.d) break;
      const ADH_GLOBAL char *p = xp[j];
      if (whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          xv[j][e] = *(const ADH_GLOBAL pt_u32 *)p;
          p += step;
        }
      } else {
        // past the last channel the address stays, and an octet without any keeps the one it loaded last
        const uint32_t c0 = ch * CHUNK + P.div_pairs.div(tid + (uint32_t)j * kPtThreads) * 8u;
        if (c0 >= P.C) p -= ch ? CHUNK * step : (size_t)0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          xv[j][e] = *(const ADH_GLOBAL pt_u32 *)p;
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
        for (int e = 0; e < 8; ++e) xv[j][e] = c0 + e < P.C ? xv[j][e] : 0u;
      }
      uintx4 v[2];
#pragma unroll
      for (int h = 0; h < (SINGLE ? 1 : 2); ++h)
#pragma unroll
        for (int d = 0; d < 4; ++d) v[h][d] = pt_pick(xv[j][2 * d], xv[j][2 * d + 1], xsel[j][h]);
      if (xat[j] != ~0u) {
        xl[xat[j]] = v[0];
        if (!SINGLE) xl[xat[j] + (SAMPLE == kDown ? P.BC + 1u : 1u)] = v[1];
      }
    }
  };

  // ---- the filter ----
  // The caller's: (output channel, WC channels of an octet) units; TAPS neighbouring elements each.
  uint32_t wv[READY ? 1 : WU][WC][WR];
  struct FilterUnit { uint32_t m, o, s; };  // output channel, octet, part of it
  auto w_unit = [&](int j) {  // forward, lanes run over the octets first: what they want then lies side by side
    const uint32_t u = tid + (uint32_t)j * kPtThreads;
    return P.flip ? FilterUnit{u % MW, u / MW / SUB, u / MW % SUB} : FilterUnit{u / SUB / OCT, u / SUB % OCT, u % SUB};
  };
  // In order: units of 16 bytes, (tap, octet) rows of MW of them.
  constexpr int RU = (TAPS * OCT * MW + kPtThreads - 1u) / kPtThreads;
  uintx4 rv[READY ? RU : 1];
  auto load_w = [&](uint32_t ch) {
    if constexpr (READY) {
      const uintx4 *base = static_cast<const uintx4 *>(P.w) + (size_t)(mg * MW / 64u * P.nchunks + ch) * (TAPS * OCT * 64u) + mg * MW % 64u;
#pragma unroll
      for (int j = 0; j < RU; ++j) {
        const uint32_t u = tid + (uint32_t)j * kPtThreads;
        if (TAPS * OCT * MW % kPtThreads != 0u && wave * 64u + (uint32_t)j * kPtThreads >= TAPS * OCT * MW) break;
        rv[j] = *(const ADH_GLOBAL uintx4 *)(base + u / MW * 64u + u % MW);
      }
    } else {
#pragma unroll
      for (int j = 0; j < WU; ++j) {
        if (SUB == 1u && wave * 64u + (uint32_t)j * kPtThreads >= WUNITS) break;
        const FilterUnit F = w_unit(j);
        const uint32_t c0 = ch * CHUNK + 8u * F.o + WC * F.s;
        const uint16_t *p = static_cast<const uint16_t *>(P.w) + (size_t)min(mg * MW + F.m, P.M - 1u) * P.w_m_stride + (size_t)min(c0, P.C - 1u) * P.w_c_stride;
        pt_load_filter<TAPS>(p, c0, P.C, P.w_c_stride, wv[j]);
      }
    }
  };
  auto store_w = [&](uint32_t ch) {
    if constexpr (READY) {
#pragma unroll
      for (int j = 0; j < RU; ++j) {
        const uint32_t u = tid + (uint32_t)j * kPtThreads;
        if (TAPS * OCT * MW % kPtThreads != 0u && wave * 64u + (uint32_t)j * kPtThreads >= TAPS * OCT * MW) break;
        wl[u] = rv[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < WU; ++j) {
        if (SUB == 1u && wave * 64u + (uint32_t)j * kPtThreads >= WUNITS) break;
        const FilterUnit F = w_unit(j);
        if ((ch + 1u) * CHUNK > P.C) pt_mask_filter(ch * CHUNK + 8u * F.o + WC * F.s, P.C, wv[j]);
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
          const auto v = pt_filter_tap(t, wv[j]);
          if constexpr (SUB == 1u) wl[((P.flip ? TAPS - 1 - t : t) * OCT + F.o) * MW + F.m] = v;
          else reinterpret_cast<std::remove_const_t<decltype(v)> *>(wl)[(((P.flip ? TAPS - 1 - t : t) * OCT + F.o) * MW + F.m) * SUB + F.s] = v;
        }
      }
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
  floatx4 acc[SETS][MT][NT];
#pragma unroll
  for (int s = 0; s < SETS; ++s)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < NT; ++q) acc[s][mt][q] = floatx4{0.f, 0.f, 0.f, 0.f};
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
    for (int t = 0; t < TAPS; ++t) {
      const uint32_t delta = tap_place(t / 3, t % 3);
#pragma unroll
      for (uint32_t ks = 0; ks < OCT / 4u; ++ks) {
        uintx4 x[NT], f[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) f[mt] = f_lane[(t * OCT + ks * 4u) * MW + mt * 16];
#pragma unroll
        for (int q = 0; q < NT; ++q) x[q] = xl[pix[q] + delta + ks * 4u * PP];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int q = 0; q < NT; ++q) acc[tap_set(t)][mt][q] = mfma_bf16(x[q], f[mt], acc[tap_set(t)][mt][q]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- results: a lane has four neighbouring pixels of a row (block widths are multiples of four) of channel 16 mt + l16 ----
  const size_t out_plane = (size_t)P.out_H * P.out_W;
  const uint32_t m0 = mg * MW + l16;
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    uint32_t b, e, r, c, tile0, n;
    P.div_live.divmod((wave * NT + q) * 16u + 4u * g, b, e);
    P.div_BC.divmod(e, r, c);
    const uint32_t img = img0 + b, i = bi * P.BR + r, j = bj * P.BC + c;
    if (b >= P.NB || img >= P.NI || i >= P.grid_VH || j >= P.grid_W) continue;
    P.div_N.divmod(img, tile0, n);
    const uint32_t t = out_tile(i);
    ADH_GLOBAL uint16_t *p = (ADH_GLOBAL uint16_t *)tab[ADH_MAX_TILES + tile0 + t] + ((size_t)n * P.M + m0) * out_plane +
                             (size_t)((i - t * P.out_step) * UP) * P.out_W + j * UP;
    const uint32_t count = min(4u, P.grid_W - j);  // (quads) of this lane that exist
    // n results side by side, some of them existing
    auto emit = [&](ADH_GLOBAL uint16_t *at, auto &v, uint32_t exist) {
      constexpr int n = sizeof(v) / sizeof(float);
      if (P.beta != 0.f) {
#pragma unroll
        for (int k = 0; k < n; ++k) v[k] += bf16_bits_to_f32(at[(uint32_t)k < exist ? k : 0]);
      }
      uint32_t pk[n / 2];
#pragma unroll
      for (int k = 0; k < n / 2; ++k) pk[k] = pt_round(v[2 * k], v[2 * k + 1]);
      if (exist == (uint32_t)n) {
        if constexpr (n == 4) *(ADH_GLOBAL pt_u32x2 *)at = uintx2{pk[0], pk[1]};
        else *(ADH_GLOBAL pt_u32x4 *)at = uintx4{pk[0], pk[1], pk[2], pk[3]};
      } else {
#pragma unroll
        for (int k = 0; k < n; ++k)
          if ((uint32_t)k < exist) at[k] = (uint16_t)(pk[k / 2] >> (k % 2 * 16));
      }
    };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (m0 + mt * 16u >= P.M) break;
      ADH_GLOBAL uint16_t *at = p + (size_t)(mt * 16) * out_plane;
      if constexpr (SAMPLE == kUp) {
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          float v[8];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            v[2 * k] = SETS == 4 ? acc[SETS == 4 ? 2 * pr : 0][mt][q][k] : pr ? 0.f : acc[0][mt][q][k];
            v[2 * k + 1] = SETS == 4 ? acc[SETS == 4 ? 2 * pr + 1 : 0][mt][q][k] : 0.f;
          }
          emit(at + (pr ? P.out_W : 0u), v, 2u * count);
        }
      } else {
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = acc[0][mt][q][k];
        emit(at, v, count);
      }
    }
  }
}

// ---- host side ----

// fp32: what `blocks` blocks of patches of `staged` pixels are expected to take, as fitted to 230 launches at stride 1 (rms error 6 %).
static double f32_patch_us(const Conv3x3Problem &q, int taps, int MT, int NT, uint32_t chunks, uint64_t blocks, uint32_t staged) {
  const bool two = taps == 1 || (MT == 1 && NT == 1 && q.sample != kDown);  // workgroups on a compute unit
  const double fit = two ? 512.0 : 256.0, rounds = std::max(1.0, 0.77 * std::ceil(blocks / fit) + 0.23 * blocks / fit);
  const double shared = two && blocks > 256u ? 1.0 + 0.336 * std::min(1.0, (blocks - 256.0) / 256.0) : 1.0;
  const double multiply = taps * (taps == 1 ? 2.0 : 1.0) * std::max(96.0 * MT * NT, 55.0 * (MT + NT));  // cycles, or operands' way out of LDS
  const double filter = (taps == 1 ? 0.17 : 0.757) * MT * (q.flip ? 0.534 : 1.0);
  return 2.8 + rounds * (1.7 + chunks * shared * (0.00096 * multiply + (taps == 1 ? 0.0053 : 0.00267) * staged + filter + 0.37));
}
// a chunk's multiplications, or their operands' way out of LDS
static double patch_multiply(int taps, uint32_t chunk, int MT, int NT) {
  return taps * (chunk / 32u) * std::max(16.0 * MT * NT, 32.0 * (MT + NT));
}
// bf16: what the launches are expected to take (see patch_plan); ready: the filter put in order first
static double bf16_patch_us(int taps, int MT, int NT, uint32_t chunks, uint64_t blocks, bool ready) {
  const double round = blocks / 512.0, full = std::min(1.0, round), multiply = patch_multiply(taps, taps == 1 ? 64u : 32u, MT, NT);
  return ready ? 3.2 + std::max(1.0, 0.6 * std::ceil(round) + 0.4 * round) * (5.9 + chunks * (0.001 * multiply * (0.033 + 1.62 * std::sqrt(full)) + 0.11 * MT))
               : 0.8 + std::ceil(round) * (3.1 + chunks * (0.00039 * multiply * (1.0 + 5.1 * std::pow(full, 1.7)) + 0.54 * MT));
}
// 3x3 at stride 1: whether no tile can be expected to take less than most_us, by its least number of blocks.  Tells large launches,
// which are the strips', without a plan.
static bool bf16_patch_exceeds(const Conv3x3Problem &q, double most_us) {
  if (most_us >= 1e30 || q.sample != kUnit) return false;
  const uint64_t pixels = (uint64_t)q.num_tiles * q.N * (q.stacked ? q.step : q.out_H) * q.out_W;
  const uint32_t chunks = (q.C + 31u) / 32u;
  for (int MT = q.M <= 16u ? 1 : q.M <= 32u ? 2 : 4; MT >= 1; MT /= 2)
    for (int NT = 4; NT >= 1; NT /= 2) {
      const uint64_t blocks = (pixels + 64u * NT - 1u) / (64u * NT) * ((q.M + 16u * MT - 1u) / (16u * MT));
      if (bf16_patch_us(9, MT, NT, chunks, blocks, false) <= most_us || bf16_patch_us(9, MT, NT, chunks, blocks, true) <= most_us) return false;
    }
  return true;
}

// Blocks of BR x BC output pixels (of NB images) by 16 MT channels, two workgroups per compute unit.  The tile is chosen by a model of
// a block's cycles: a chunk's multiplications (or their operands' way out of LDS), its staging, and a load's latency.
// Whether the filter is put in order first, is decided by times as fitted to 566 shapes, rounds of 512 workgroups of n chunks each,
// `multiply` cycles of matrix work a chunk, f the part of a round's workgroups that exist:
//   the caller's filter        rounds (4.1 + n (0.00032 multiply (1 + 5.3 f) + 0.52 MT)) us
//   put in order first   2.1 + rounds (5.4 + n 0.00096 multiply (1 + 1.06 f)) us
// (from 20 us on the second: forward, the caller's filter costs a line of cache per lane and load.  64 -> 64 channels, 8 tiles of
// 128 x 2048 717 -> 578 us, 16 -> 32 on 72 x 16 4.7 -> 7.3.)  The launch's time is then expected as fitted to 5000 passes served here (bf16_patch_us;
// rms error 14 %): a round that is begun takes most of a whole one's time.
int patch_plan(const Conv3x3Problem &q, int taps, int parts, size_t workspace_bytes, PatchPlan *plan) {
  PatchParams &P = plan->P;
  P.N = q.N; P.C = q.C; P.M = q.M; P.num_tiles = q.num_tiles;
  P.NI = q.stacked ? q.N : q.N * q.num_tiles;
  P.in_H = q.in_H; P.in_W = q.in_W; P.out_H = q.out_H; P.out_W = q.out_W;
  if (q.in_W < 2u) return ADH_EUNIMPL;
  P.in_VH = q.in_H; P.grid_VH = q.sample == kUp ? q.in_H : q.out_H; P.grid_W = q.sample == kUp ? q.in_W : q.out_W;
  P.in_step = q.in_H; P.out_step = q.out_H;
  if (q.stacked) {
    if ((uint64_t)q.step * q.num_tiles * (q.sample == kUnit ? 1u : 2u) + 2u >= (1ull << 31)) return ADH_EUNIMPL;
    P.in_lead = q.in_lead; P.out_lead = q.out_lead;
    P.in_step = P.out_step = q.step;
    if (q.sample == kDown) P.in_step = 2u * q.step;
    P.in_VH = P.in_step * q.num_tiles + 2u * q.in_lead;
    P.grid_VH = q.step * q.num_tiles + 2u * q.out_lead;
    P.last_tile = q.num_tiles - 1u;
  }
  P.w_m_stride = q.w_m_stride; P.w_c_stride = q.w_c_stride;
  P.pad_r = q.pad_r; P.pad_c = q.pad_c; P.dil = q.dil; P.flip = q.flip ? 1 : 0;
  P.beta = q.beta;
  const uint32_t chunk = taps == 1 ? 64u : 32u;
  P.nchunks = (P.C + chunk - 1u) / chunk;
  // rows of n output rows' patch; pairs and pixels of a row of n output columns
  auto rows_of = [&](uint32_t n) { return taps == 1 ? n : q.sample == kDown ? 2u * n + 1u : q.sample == kUp ? n + 1u : n + 2u * q.dil; };
  auto pairs_of = [&](uint32_t n) { return q.sample == kDown ? (taps == 1 ? n : n + 1u) : taps == 1 ? n / 2u : q.sample == kUp ? n / 2u + 1u : n / 2u + q.dil; };
  const uint32_t per_pair = q.sample == kDown && taps == 1 ? 1u : 2u;
  double best = 1e300;
  uint32_t nbi = 0, nbj = 0;
  const uint64_t grid_pixels = (uint64_t)P.NI * P.grid_VH * P.grid_W;
  // what `blocks` blocks of patches of `staged` pixels cost: a chunk's staging is instructions per unit, and its way through the cache
  auto price = [&](int MT, int NT, uint64_t blocks, uint32_t staged) {
    if (parts == 3) return f32_patch_us(q, taps, MT, NT, P.nchunks, blocks, staged);
    const double multiply = patch_multiply(taps, chunk, MT, NT), stage = 300.0 + 0.6 * staged + 4.0 * taps * MT;
    const double alone = 5000.0 + P.nchunks * (multiply + stage + 1000.0), both = 3000.0 + P.nchunks * std::max(2.0 * multiply + stage, multiply + stage + 1000.0);
    return (blocks <= 256u ? alone : std::max(alone, (double)((blocks + 511u) / 512u) * both)) + 1e-3 * (double)blocks;
  };
  // The tiles by what they cost with their least number of blocks, so that most are passed over (the plan is made anew on every call:
  // 16 -> 16 channels on 2 tiles of 4 x 2000 1.2 -> 0.5 us of host time, with the same choices).
  struct Tile { double least; int MT, NT; } tiles[9];
  int num_tiles = 0;
  for (int MT = P.M <= 16u ? 1 : P.M <= 32u || parts == 3 ? 2 : 4; MT >= 1; MT /= 2)
    for (int NT = parts == 3 ? (q.sample == kUnit || taps == 1 ? 2 : 1) : q.sample == kUnit || taps == 1 ? 4 : 2; NT >= 1; NT /= 2) {
      const uint32_t slots = 64u * NT;
      const Tile tile = {price(MT, NT, (grid_pixels + slots - 1u) / slots * ((P.M + 16u * MT - 1u) / (16u * MT)), (uint32_t)std::min<uint64_t>(slots, grid_pixels)), MT, NT};
      int k = num_tiles++;
      for (; k > 0 && tiles[k - 1].least > tile.least; --k) tiles[k] = tiles[k - 1];
      tiles[k] = tile;
    }
  for (int k = 0; k < num_tiles && tiles[k].least < best; ++k) {
    const int MT = tiles[k].MT, NT = tiles[k].NT;
    const uint32_t MG = (P.M + 16u * MT - 1u) / (16u * MT), slots = 64u * NT, pixels = pt_pixels(q.sample, taps, NT, parts);
    uint32_t last_BC = 0;
    for (uint32_t cuts = (P.grid_W + slots - 1u) / slots; cuts <= P.grid_W; cuts += 1u + cuts / 4u) {
      const uint32_t BC = ((P.grid_W + cuts - 1u) / cuts + 3u) & ~3u;
      if (cuts > 1u && BC < 8u) break;
      const uint32_t pitch = pairs_of(BC) * per_pair;
      if (BC > slots || BC == last_BC || rows_of(1u) * pitch > pixels) continue;
      last_BC = BC;
      // (rows_of is linear)
      const uint32_t held = pixels / pitch, one = rows_of(1u), more = rows_of(2u) - one;
      const uint32_t max_BR = std::min(std::min(P.grid_VH, slots / BC), 1u + (held - one) / more);
      const uint32_t nc = (P.grid_W + BC - 1u) / BC, nr = (P.grid_VH + max_BR - 1u) / max_BR, BR = (P.grid_VH + nr - 1u) / nr;
      const uint32_t image = rows_of(BR) * pitch;
      uint32_t NB = std::min(std::min(slots / (BR * BC), pixels / image), P.NI);
      const uint32_t groups = (P.NI + NB - 1u) / NB;
      NB = (P.NI + groups - 1u) / groups;
      const uint64_t blocks = (uint64_t)groups * nc * nr * MG;
      const double cost = price(MT, NT, blocks, NB * image);
      if (cost >= best) continue;
      best = cost;
      plan->MT = MT; plan->NT = NT;
      P.BR = BR; P.BC = BC; P.NB = NB; P.pitch = pitch; P.image = image;
      nbi = nr; nbj = nc;
    }
  }
  if (nbi == 0u) return ADH_EUNIMPL;
  const uint32_t MG = (P.M + 16u * plan->MT - 1u) / (16u * plan->MT), pairs = P.NB * P.image / per_pair;
  const uint64_t blocks = (uint64_t)((P.NI + P.NB - 1u) / P.NB) * nbi * nbj * MG;
  if (blocks >= (1ull << 23)) return ADH_EUNIMPL;  // (threads of a launch)
  P.blocks = (uint32_t)blocks;
  P.xcd_chunk = (P.blocks + 7u) / 8u;
  P.div_bpg = FastDiv(nbi * nbj); P.div_nbj = FastDiv(nbj); P.div_MG = FastDiv(MG); P.div_N = FastDiv(P.N);
  P.div_BC = FastDiv(P.BC); P.div_live = FastDiv(P.BR * P.BC);
  P.div_pairs = FastDiv(pairs); P.div_pairs_img = FastDiv(P.image / per_pair); P.div_pairs_row = FastDiv(P.pitch / per_pair);
  P.div_in = FastDiv(P.in_step); P.div_out = FastDiv(P.out_step);
  if (parts == 3) {
    plan->us = best;
    return ADH_OK;
  }
  const double full = std::min(1.0, blocks / 512.0), rounds = std::max(1.0, blocks / 512.0), multiply = patch_multiply(taps, chunk, plan->MT, plan->NT);
  const double first_us = 2.1 + rounds * (5.4 + P.nchunks * 0.00096 * multiply * (1.0 + 1.06 * full));
  plan->units = (uint64_t)((P.M + 63u) / 64u) * P.nchunks * 256u;
  plan->ready = taps == 9 && first_us < rounds * (4.1 + P.nchunks * (0.00032 * multiply * (1.0 + 5.3 * full) + 0.52 * plan->MT)) &&
                plan->units * 144u <= workspace_bytes && plan->units < (1ull << 31);
  plan->us = bf16_patch_us(taps, plan->MT, plan->NT, P.nchunks, blocks, plan->ready);
  return ADH_OK;
}

template <int MT, int NT, int SAMPLE, int TAPS>
static void launch_patch(const PatchPlan &plan, hipStream_t st) {
  const dim3 grid(plan.P.xcd_chunk * 8u), block(kPtThreads);
  if constexpr (TAPS == 9) {
    if (plan.ready) {
      hipLaunchKernelGGL((conv_bf16_patch_kernel<MT, NT, SAMPLE, TAPS, true>), grid, block, 0, st, plan.P);
      return;
    }
  }
  hipLaunchKernelGGL((conv_bf16_patch_kernel<MT, NT, SAMPLE, TAPS, false>), grid, block, 0, st, plan.P);
}
template <int MT, int SAMPLE, int TAPS>
static void launch_patch_nt(const PatchPlan &plan, hipStream_t st) {
  if constexpr (SAMPLE == kUnit || TAPS == 1) {
    if (plan.NT == 4) return launch_patch<MT, 4, SAMPLE, TAPS>(plan, st);
  }
  if (plan.NT == 2) launch_patch<MT, 2, SAMPLE, TAPS>(plan, st);
  else launch_patch<MT, 1, SAMPLE, TAPS>(plan, st);
}
template <int SAMPLE, int TAPS>
static void launch_patch_mt(const PatchPlan &plan, hipStream_t st) {
  if (plan.MT == 4) launch_patch_nt<4, SAMPLE, TAPS>(plan, st);
  else if (plan.MT == 2) launch_patch_nt<2, SAMPLE, TAPS>(plan, st);
  else launch_patch_nt<1, SAMPLE, TAPS>(plan, st);
}

bool conv_bf16_patch_name(const Conv3x3Problem &q, int taps, size_t workspace_bytes, double most_us, char *name, size_t name_bytes) {
  PatchPlan plan = {};
  if (bf16_patch_exceeds(q, most_us) || patch_plan(q, taps, 1, workspace_bytes, &plan) || plan.us > most_us) return false;
  snprintf(name, name_bytes, "conv_bf16_patch_kernel<%d, %d, %d, %d, %s>", plan.MT, plan.NT, (int)q.sample, taps, plan.ready ? "true" : "false");
  return true;
}

int conv_bf16_patch(const Conv3x3Problem &q, int taps, void *workspace, size_t workspace_bytes, double most_us, hipStream_t st) {
  if (bf16_patch_exceeds(q, most_us)) return ADH_EUNIMPL;
  PatchPlan plan = {};
  const int e = patch_plan(q, taps, 1, workspace ? workspace_bytes : 0u, &plan);
  if (e) return e;
  if (plan.us > most_us) return ADH_EUNIMPL;
  for (uint32_t t = 0; t < q.num_tiles; ++t) {
    plan.P.in[t] = q.in[t];
    plan.P.out[t] = q.out[t];
  }
  plan.P.w = q.w;
  if (plan.ready) {
    hipLaunchKernelGGL(conv_bf16_patch_filter_kernel, dim3((uint32_t)((plan.units + kPtThreads - 1u) / kPtThreads)), dim3(kPtThreads), 0, st, reinterpret_cast<const uint16_t *>(q.w),
                       reinterpret_cast<uintx4 *>(workspace), plan.P.M, plan.P.C, plan.P.nchunks, plan.P.w_m_stride, plan.P.w_c_stride, plan.P.flip,
                       (uint32_t)plan.units);
    plan.P.w = workspace;
  }
  if (taps == 9) {
    if (q.sample == kUnit) launch_patch_mt<kUnit, 9>(plan, st);
    else if (q.sample == kDown) launch_patch_mt<kDown, 9>(plan, st);
    else launch_patch_mt<kUp, 9>(plan, st);
  } else {
    if (q.sample == kUnit) launch_patch_mt<kUnit, 1>(plan, st);
    else if (q.sample == kDown) launch_patch_mt<kDown, 1>(plan, st);
    else launch_patch_mt<kUp, 1>(plan, st);
  }
  return launch_status();
}

}  // namespace adh
