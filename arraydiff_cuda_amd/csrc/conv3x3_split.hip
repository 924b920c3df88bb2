// 3x3 convolution at stride 1 in fp32 on the bf16 matrix cores (split_bf16.h says how), forward and backward-data over
// halo-padded tiles and over tiles without halo:
//   out[m][R][Q] = beta*out + sum over c, a, b of w[m][c][a][b] * in[c][R + D*a - pad_r][Q + D*b - pad_c]
//
// Mapping.  v_mfma_f32_16x16x32_bf16, k = 32 channels of one tap (register-fed it sustains 2.26 PFLOP/s here, the 32x32x16
// form 1.98: half the accumulator traffic per flop).  A workgroup of eight waves, one per compute unit, owns 16*MT output
// channels of 128*NT output pixels; a wave all of the channels and 16*NT of the pixels.  At MT = NT = 4 a step (a tap of a
// chunk of 32 channels) reads 24 operands of 1 KB per wave and issues 96 MFMAs: half of the LDS bandwidth.
//   * The input patch of a chunk is staged once, split into its parts, as [part][octet of channels][pixel][8 channels]: an
//     operand is one ds_read_b128 of neighbouring pixels whatever the tap.  The next chunk's elements are loaded into
//     registers during the steps and split and stored at the chunk's end (122 KB of LDS: a second buffer does not fit).
//   * The filter is read as the caller holds it and split on the way to LDS, tap by tap, two steps ahead, into a ring of
//     three slots: one barrier a step, and the first operands of a step are fetched in the one before.
//   * What a step has to do besides multiplying is dealt out between its groups of NT MFMAs.  Done in one piece at the
//     step's start, both waves of a SIMD stood in it at once (212 TFLOP/s, 256 channels on 8 x 32 tiles; 232 dealt out).
//   * The products below h*h are summed apart from it, or for some taps, as the registers allow (LOW below): additions at the
//     size of the whole sum, six a tap, would cost digits that fp32 sums have.
//   * The workgroups are persistent and the sequence of chunks runs on across their blocks: the next block's first patch
//     and filter rows arrive during the last steps of this one.
// Row tiles of one tensor are addressed as that tensor: a patch row is divided by the tile height to find its tile, so a
// workgroup may span tiles (a 4 x 16 tile is a quarter of a 16 x 16 image) and no halo exchange or reduction is needed.
//
// Measured at stride 2 (32 images, 4 tiles, forward / backward-data; v_mfma_f32 kernels before): 64 -> 128 channels on 32 x 128
// tiles 0.214 -> 0.188 / 0.212 -> 0.130 ms, 128 -> 256 on 16 x 64 0.205 -> 0.182 / 0.192 -> 0.118 (163 TFLOP/s), 256 -> 512 on
// 8 x 32 0.206 -> 0.179 / 0.187 -> 0.132; 48 channels on 3 tiles of 6 x 30 0.023 -> 0.013 / 0.019 -> 0.014.  A forward step has a
// quarter of the stride-1 step's products and the same patch to load and split: that bounds it.  The next patch's loads go out
// from the chunk's first step on (stride 1 has the registers for them from the fourth): 0.202 -> 0.187 and 0.126 -> 0.118.
// Measured (32 images, 4 tiles without halo, forward / backward-data; v_mfma_f32 kernels before): 64 channels on 32 x 128
// tiles 0.309 -> 0.209 / 0.197 ms (196 TFLOP/s), 128 on 16 x 64 0.297 -> 0.182, 256 on 8 x 32 0.292 -> 0.175 (221), 512 on
// 4 x 16 0.39 -> 0.215 / 0.212; with the arguments read where they are used (from_memory; 130 to 200 scalar registers were spilled) 512 on 4 x 16
// 0.246 -> 0.237, backward-data at stride 2, 128 -> 256 on 16 x 64, 0.131 -> 0.120, 60 random padded layers 0.967 / 0.974 of the time, up to
// 0.88 where a block has 32 channels.  Bound: the matrix pipe is busy 0.6 of the cycles; a step of 3072 matrix cycles takes 3700 to 4400
// (the loads' address arithmetic and the splitting compete for issue slots), the patch's change of chunk 4500, and a block's
// results leave at the rate of the memory, all workgroups at once.
#include "conv3x3_split.h"

#include <stdio.h>

#include <algorithm>
#include <utility>

#include "split_bf16.h"

namespace adh {

constexpr uint32_t kSpThreads = 512;
constexpr uint32_t kSpChunk = 32;  // channels per staged chunk
constexpr uint32_t kSpPP = 640;    // patch pixels per plane in LDS
// a block's patch pixels; quads have few (and four sets of sums: what is staged for more pixels would be spilled)
constexpr uint32_t split_patch(int sample) { return sample == kUp ? 384u : kSpPP; }
constexpr int kLowApart = 10;
constexpr uint32_t kSpMP = 68;     // filter rows per plane: = 4 (mod 16), so that the octet planes start 64 bytes apart

struct SplitParams {
  const float *in[ADH_MAX_TILES];
  const float *res[ADH_MAX_TILES];  // what beta adds: the output itself or a residual laid out like it
  float *out[ADH_MAX_TILES];
  const float *w;
  float *part;  // ksplit > 1: sums, [split][tile] laid out like an output tile
  uint64_t part_tile_elems;
  uint32_t N, NI, C, M, num_tiles;
  uint32_t in_H, in_W, out_H, out_W;
  uint32_t in_VH, grid_VH, grid_W;  // rows of the (stacked) input; what the blocks tile: output pixels, or quads of them
  uint32_t in_lead, out_lead, in_step, out_step, last_tile;
  uint32_t w_m_stride, w_c_stride;
  uint32_t BR, BC, NB, PPn;  // a block's pixels: BR x BC of NB images; patch pixels
  uint32_t nchunks, chunks_per_split, ksplit, blocks, xcd_chunk;
  int32_t pad_r, pad_c, flip;
  uint32_t dil;
  float beta;
  FastDiv div_bpg, div_nbj, div_MG, div_N, div_BC, div_live, div_PPI, div_PCP, div_PPn, div_ksplit, div_in, div_out;
};

__device__ __forceinline__ floatx4 load4(const ADH_GLOBAL float *p) { return *(const ADH_GLOBAL floatx4_u *)p; }
__device__ __forceinline__ void store4(ADH_GLOBAL float *p, floatx4 v) { *(ADH_GLOBAL floatx4_u *)p = v; }

template <int... I, typename F>
__device__ __forceinline__ void static_for_seq(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(0), f(1), .. with the index a compile-time constant
template <int N, typename F>
__device__ __forceinline__ void static_for(F f) {
  static_for_seq(std::make_integer_sequence<int, N>{}, f);
}

// A block of the launch: which output channels, pixels and channel chunks.
struct SplitBlock {
  uint32_t mg, img0, bi, bj, ks, ch_lo, ch_hi;
};

// VEC: a lane's results are four neighbouring pixels of one channel (pixels on the matrix rows), stored 16 bytes at a time:
// block and output widths are multiples of four.  Otherwise four channels of one pixel, whose stores are runs of 16 pixels.
//
// SAMPLE.  Stride 2, padding 1 (tiles of even height and width):
//   kDown, forward: the patch is (2 BR + 1) x (2 BC + 1), a row's even columns first, so that the 16 pixels of an operand are
//     neighbours in LDS for every tap.  640 patch pixels leave 128 output pixels to a block (NT = 1).
//   kUp, backward-data: a block owns quads, the 2 x 2 gradient pixels at (2i, 2j), which tap (1 +- a, 1 +- b) of the filter feeds
//     from dy[i .. i + 1][j .. j + 1]: nine taps over a patch of (BR + 1) x (BC + 1), into four sets of sums.  A lane's four
//     neighbouring quads are two rows of eight pixels.
//
// LOW.  Six products of parts go into a sum per tap and chunk, and each addition is rounded at the size of the sum; all but h*h
// are below 2^-8 of it.  kLowApart: they have sums of their own, added at the block's end, and cost no digit.  Where registers
// are short, the small products of LOW of the nine taps are summed up from zero and added at once; 0: every product is added
// by itself.  The choice hangs on the channels alone, not on the block's shape or the images it holds (split_low); small launches go
// to conv_f32_patch.hip, which adds in another order: the forms of one layer have the same bits, not a layer and a part of it.
template <int MT, int NT, bool VEC, int SAMPLE, int LOW>
__global__ __launch_bounds__(kSpThreads, 2) void conv3x3_split_kernel(const SplitParams args) {
  const SplitParams &P = args;
  constexpr uint32_t MW = 16u * MT;
  constexpr int SETS = SAMPLE == kUp ? 4 : 1;  // of sums
  constexpr uint32_t DOWN = SAMPLE == kDown ? 2u : 1u, UP = SAMPLE == kUp ? 2u : 1u;
  constexpr uint32_t SLOT = 3 * 4 * kSpMP;  // the operands of a tap
  constexpr int XU = (4 * split_patch(SAMPLE) + kSpThreads - 1) / kSpThreads;  // (pixel, octet) units a thread stages
  __shared__ __align__(16) uintx4 xl[3 * 4 * kSpPP];
  __shared__ __align__(16) uintx4 wl[3 * SLOT];
  __shared__ const float *tab[3 * ADH_MAX_TILES];  // the tiles' addresses: in, out, res
  __shared__ uint32_t not_finite;
  constexpr bool APART = LOW == kLowApart;
  constexpr int FIRST = SAMPLE == kUnit ? 3 : 0;  // step whose side work loads the next patch's first unit
  const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));

  // neighbouring blocks (the channel groups of one block of pixels first) run on one XCD and share its cache
  const uint32_t per_xcd = gridDim.x >> 3;
  uint32_t next_vid = (blockIdx.x & 7u) * P.xcd_chunk + (blockIdx.x >> 3);
  const uint32_t end_vid = min(P.blocks, ((blockIdx.x & 7u) + 1u) * P.xcd_chunk);
  if (next_vid >= end_vid) return;
  auto next_block = [&]() {
    const SplitParams &P = from_memory(args);
    SplitBlock B;
    uint32_t bid, outer, inner, group;
    P.div_ksplit.divmod(next_vid, bid, B.ks);
    next_vid += per_xcd;
    P.div_MG.divmod(bid, outer, B.mg);
    P.div_bpg.divmod(outer, group, inner);
    P.div_nbj.divmod(inner, B.bi, B.bj);
    B.ch_lo = B.ks * P.chunks_per_split;
    B.ch_hi = min(P.nchunks, B.ch_lo + P.chunks_per_split);
    B.img0 = group * P.NB;
    return B;
  };

  // (a per-lane choice of tile would be looked up one lane group at a time from the kernel's arguments)
  if (tid < P.num_tiles) {
    tab[tid] = P.in[tid];
    tab[ADH_MAX_TILES + tid] = P.out[tid];
    tab[2 * ADH_MAX_TILES + tid] = P.res[tid];
  }
  if (tid == 0u) not_finite = 0u;
  lds_barrier();

  // tile of row R of the stacked tensor
  auto in_tile = [&](const SplitParams &P, uint32_t R) { return R < P.in_lead ? 0u : min(P.div_in.div(R - P.in_lead), P.last_tile); };
  auto out_tile = [&](const SplitParams &P, uint32_t R) { return R < P.out_lead ? 0u : min(P.div_out.div(R - P.out_lead), P.last_tile); };

  // ---- the patch: this thread stages units tid + j * kSpThreads of its pixels' octets (octet 0 of all pixels first);
  // element e of octet o is channel 4e + o of the chunk, the filter's order below ----
  const size_t plane = (size_t)P.in_H * P.in_W;
  float xv[XU][8];
  uint32_t xn = 0;  // four bits a unit: how many of its elements exist
  // (hidden from the compiler, which would keep everything it can derive from the thread's index in registers)
  auto unit = [&](int j) {
    uint32_t u = tid + (uint32_t)j * kSpThreads;
    asm volatile("" : "+v"(u));
    return u;
  };
  auto idle = [&](int j) {  // of the wave's units
    uint32_t u = (uint32_t)j * kSpThreads + wave * 64u;
    asm volatile("" : "+s"(u));
    return u >= 4u * P.PPn;
  };
  const ADH_GLOBAL char *src = nullptr;  // the next element to load, and how many there are of the unit
  uint32_t src_n = 0;
  auto set_unit = [&](const SplitBlock &B, uint32_t ch, int j) {
    const SplitParams &P = from_memory(args);
    uint32_t o, p, b, e, r, c;
    P.div_PPn.divmod(unit(j), o, p);
    P.div_PPI.divmod(p, b, e);
    P.div_PCP.divmod(e, r, c);
    if constexpr (SAMPLE == kDown) c = c <= P.BC ? 2u * c : 2u * (c - P.BC) - 1u;
    const uint32_t img = B.img0 + b, c0 = ch * kSpChunk + o;
    const int32_t R = (int32_t)(B.bi * P.BR * DOWN + r) - P.pad_r, Q = (int32_t)(B.bj * P.BC * DOWN + c) - P.pad_c;
    const bool ok = o < 4u && c0 < P.C && img < P.NI && R >= 0 && R < (int32_t)P.in_VH && Q >= 0 && Q < (int32_t)P.in_W;
    uint32_t tile0, n;
    P.div_N.divmod(ok ? img : 0u, tile0, n);
    const uint32_t Ru = ok ? (uint32_t)R : P.in_lead, t = in_tile(P, Ru);
    src_n = ok ? min(8u, (P.C - c0 + 3u) >> 2) : 0u;
    xn = (j == 0 ? 0u : xn) | src_n << (4 * j);
    // (a unit that does not exist loads an existing place; its values are replaced by zero)
    src = (const ADH_GLOBAL char *)tab[tile0 + t] +
          (((size_t)n * P.C + (ok ? c0 : 0u)) * plane + (size_t)(Ru - t * P.in_step) * P.in_W + (ok ? (uint32_t)Q : 0u)) * 4u;
  };
  auto load_elems = [&](int j, int e0, int e1) {  // elements [e0, e1) of unit j
#pragma unroll
    for (int e = e0; e < e1; ++e) {
      xv[j][e] = *(const ADH_GLOBAL float *)src;
      // past the last channel the address stays; (it walks because eight addresses at once would not fit the registers)
      src += (uint32_t)(e + 1) < src_n ? 16u * plane : (size_t)0;
      asm("" : "+v"(src));
    }
  };
  auto store_x = [&]() {
    const SplitParams &P = from_memory(args);
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < XU; ++j) {
      if (idle(j)) break;
      uint32_t o, p;
      P.div_PPn.divmod(unit(j), o, p);
      const uint32_t n = xn >> (4 * j) & 15u;
      if (__builtin_amdgcn_ballot_w64(n < 8u)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[j][e] = (uint32_t)e < n ? xv[j][e] : 0.f;
      }
      uintx4 part[3];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint32_t h, m, l;
        mx = max_abs(mx, xv[j][2 * q], xv[j][2 * q + 1]);
        split_pair(xv[j][2 * q], xv[j][2 * q + 1], h, m, l);
        part[0][q] = h; part[1][q] = m; part[2][q] = l;
      }
      if (o < 4u) {
#pragma unroll
        for (int k = 0; k < 3; ++k) xl[(k * 4 + o) * kSpPP + p] = part[k];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (mx >= kSplitLimit) not_finite = 1u;
  };
  // The staged values' loads have been waited for when this is passed: done ahead of a block's stores, which the wait
  // would otherwise take in.
  auto settle_x = [&]() {
#pragma unroll
    for (int j = 0; j < XU; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(xv[j][e]));
  };

  // ---- the filter: thread (m, half octet) of the block's MW x 8 loads four channels x three taps of a filter row.
  // Forward, lanes run over the octets first: what they want of the caller's [m][c][tap] then shares cache lines. ----
  struct FilterLane { uint32_t oct, m, half; };
  auto w_lane = [&]() {
    uint32_t u = tid;
    asm volatile("" : "+v"(u));  // (as above)
    return P.flip ? FilterLane{(u / MW) & 3u, u % MW, u / (4u * MW)} : FilterLane{u & 3u, (u >> 2) % MW, u / (4u * MW)};
  };
  float wrow[12];
  auto load_wrow = [&](uint32_t mg, uint32_t ch, int kh) {
    const SplitParams &P = from_memory(args);
    const FilterLane L = w_lane();
    const float *base = P.w + (size_t)min(mg * MW + L.m, P.M - 1u) * P.w_m_stride + (P.flip ? 6 - 3 * kh : 3 * kh);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float *p = base + (size_t)min(ch * kSpChunk + 4u * (4u * L.half + e) + L.oct, P.C - 1u) * P.w_c_stride;
#pragma unroll
      for (int b = 0; b < 3; ++b) wrow[e * 3 + b] = p[b];
    }
  };
  // (what a reduction channel that does not exist multiplies is zero, and a produced one is dropped: nothing is masked here)
  uint32_t wpart[3][2];
  float w_mx = 0.f;
  auto pack_w = [&](int b, int q) {  // channels 2q, 2q + 1 of column b of the filter row in wrow
    const float v0 = P.flip ? wrow[6 * q + 2 - b] : wrow[6 * q + b], v1 = P.flip ? wrow[6 * q + 5 - b] : wrow[6 * q + 3 + b];
    w_mx = max_abs(w_mx, v0, v1);
    split_pair(v0, v1, wpart[0][q], wpart[1][q], wpart[2][q]);
  };
  auto store_w = [&](uint32_t slot) {
    const FilterLane L = w_lane();
    if (L.half < 2u) {
#pragma unroll
      for (int k = 0; k < 3; ++k)
        reinterpret_cast<uintx2 *>(wl + slot * SLOT + (k * 4 + L.oct) * kSpMP + L.m)[L.half] = uintx2{wpart[k][0], wpart[k][1]};
    }
    if (w_mx >= kSplitLimit) not_finite = 1u;
  };

  // ---- this wave's pixels: 16 consecutive ones of the block's NB x BR x BC per tile ----
  uint32_t pix[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    uint32_t b, e, r, c;
    P.div_live.divmod((wave * NT + q) * 16u + l16, b, e);
    P.div_BC.divmod(e, r, c);
    pix[q] = (b < P.NB ? b * P.div_PPI.d + r * DOWN * P.div_PCP.d + c : 0u) + g * kSpPP;
  }
  // where a tap of the window lies in the patch, and the set of sums that it feeds
  auto tap_place = [&](uint32_t a, uint32_t b) {
    if constexpr (SAMPLE == kDown) return a * P.div_PCP.d + (b == 1u ? P.BC + 1u : b / 2u);
    else if constexpr (SAMPLE == kUp) return a / 2u * P.div_PCP.d + b / 2u;
    else return (a * P.div_PCP.d + b) * P.dil;
  };
  auto tap_set = [](int t) { return SAMPLE == kUp ? (t / 3 == 1 ? 0 : 2) + (t % 3 == 1 ? 0 : 1) : 0; };
  floatx4 acc[SETS][MT][NT];
  floatx4 low[APART ? SETS : 1][APART ? MT : 1][NT];
  const uintx4 *const a_lane = wl + g * kSpMP + l16;

  // ---- results ----
  const size_t out_plane = (size_t)P.out_H * P.out_W;
  struct Place { bool ok; uint32_t img, i, j, tile; size_t at; };
  auto place_of = [&](const SplitBlock &B, uint32_t f) {  // pixel slot f of the block
    const SplitParams &P = from_memory(args);
    Place pl;
    uint32_t b, e, r, c, tile0, n;
    asm volatile("" : "+v"(f));  // (worked out where it is used, not kept)
    P.div_live.divmod(f, b, e);
    P.div_BC.divmod(e, r, c);
    pl.img = B.img0 + b;
    pl.i = B.bi * P.BR + r;
    pl.j = B.bj * P.BC + c;
    pl.ok = b < P.NB && pl.img < P.NI && pl.i < P.grid_VH && pl.j < P.grid_W;
    P.div_N.divmod(pl.ok ? pl.img : 0u, tile0, n);
    const uint32_t R = pl.ok ? pl.i : P.out_lead, t = out_tile(P, R);
    pl.tile = tile0 + t;
    pl.at = (size_t)n * P.M * out_plane + (size_t)((R - t * P.out_step) * UP) * P.out_W + (pl.ok ? pl.j * UP : 0u);
    return pl;
  };
  auto emit_all = [&](const SplitBlock &B) {
    const SplitParams &P = from_memory(args);
    // channel of accumulator (mt, i) above m0: 16 mt (VEC) or 16 mt + i
    const uint32_t m0 = B.mg * MW + (VEC ? l16 : g * 4u), m_top = P.M - 1u - min(m0, P.M - 1u);
    const bool whole = (B.mg + 1u) * MW <= P.M;
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      const Place pl = place_of(B, (wave * NT + q) * 16u + (VEC ? 4u * g : l16));
      if (!pl.ok) continue;
      const size_t o = pl.at + (size_t)m0 * out_plane;
      const bool sums = P.ksplit > 1u;
      ADH_GLOBAL float *p = (ADH_GLOBAL float *)(sums ? P.part + ((size_t)B.ks * P.num_tiles + pl.tile) * P.part_tile_elems
                                                      : const_cast<float *>(tab[ADH_MAX_TILES + pl.tile])) + o;
      if constexpr (SAMPLE == kUp) {
        const bool adds = !sums && P.beta != 0.f;
        const ADH_GLOBAL float *r = (const ADH_GLOBAL float *)tab[2 * ADH_MAX_TILES + pl.tile] + o;
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          const size_t row = pr ? (size_t)P.out_W : 0u;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const floatx4 even = acc[2 * pr][mt][q], odd = acc[2 * pr + 1][mt][q];
            if constexpr (VEC) {
              if (!whole && m0 + mt * 16u >= P.M) continue;
              const size_t at = (size_t)(mt * 16) * out_plane + row;
              floatx4 lo = {even[0], odd[0], even[1], odd[1]}, hi = {even[2], odd[2], even[3], odd[3]};
              if (adds) {
                lo += load4(r + at);
                hi += load4(r + at + 4);
              }
              store4(p + at, lo);
              store4(p + at + 4, hi);
            } else {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                if (!whole && m0 + mt * 16u + i >= P.M) continue;
                const size_t at = (size_t)(mt * 16 + i) * out_plane + row;
                p[at] = adds ? even[i] + r[at] : even[i];
                p[at + 1] = adds ? odd[i] + r[at + 1] : odd[i];
              }
            }
          }
        }
        continue;
      }
      if (!sums && P.beta != 0.f) {
        // (channels that do not exist read an existing one)
        const ADH_GLOBAL float *r = (const ADH_GLOBAL float *)tab[2 * ADH_MAX_TILES + pl.tile] + (pl.at + (size_t)min(m0, P.M - 1u) * out_plane);
        floatx4 old[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          if constexpr (VEC) {
            old[mt] = load4(r + (size_t)min(mt * 16u, m_top & ~15u) * out_plane);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) old[mt][i] = r[(size_t)min(mt * 16u + i, m_top) * out_plane];
          }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[0][mt][q] += old[mt];
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if constexpr (VEC) {
          if (whole || m0 + mt * 16u < P.M) store4(p + (size_t)(mt * 16) * out_plane, acc[0][mt][q]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (whole || m0 + mt * 16u + i < P.M) p[(size_t)(mt * 16 + i) * out_plane] = acc[0][mt][q][i];
        }
      }
    }
  };
  // something staged has parts that are not finite: the wave's outputs as plain fp32 sums, straight from memory
  auto emit_plain = [&](const SplitBlock &B) {
    const SplitParams &P = from_memory(args);
    for (uint32_t of = lane; of < 16u * NT * MW * SETS; of += 64u) {
      const uint32_t at = of / SETS, set = of % SETS, m = B.mg * MW + at / (16u * NT);
      const Place pl = place_of(B, wave * (16u * NT) + at % (16u * NT));
      if (!pl.ok || m >= P.M) continue;
      uint32_t tile0, n;
      P.div_N.divmod(pl.img, tile0, n);
      float v = 0.f;
      for (uint32_t c = B.ch_lo * kSpChunk; c < min(B.ch_hi * kSpChunk, P.C); ++c)
        for (uint32_t t = 0; t < 9u; ++t) {
          if (SAMPLE == kUp && (uint32_t)tap_set((int)t) != set) continue;
          const uint32_t a = SAMPLE == kUp ? t / 6u : t / 3u, b = SAMPLE == kUp ? t % 3u / 2u : t % 3u;
          const int32_t R = (int32_t)(pl.i * DOWN + a * P.dil) - P.pad_r, Q = (int32_t)(pl.j * DOWN + b * P.dil) - P.pad_c;
          float x = 0.f;  // the padding is data: an infinite filter element times it is NaN
          if (R >= 0 && R < (int32_t)P.in_VH && Q >= 0 && Q < (int32_t)P.in_W) {
            const uint32_t ti = in_tile(P, (uint32_t)R);
            x = tab[tile0 + ti][((size_t)n * P.C + c) * plane + ((uint32_t)R - ti * P.in_step) * (size_t)P.in_W + (uint32_t)Q];
          }
          v = __builtin_fmaf(P.w[(size_t)m * P.w_m_stride + (size_t)c * P.w_c_stride + (P.flip ? 8u - t : t)], x, v);
        }
      const size_t o = pl.at + (size_t)m * out_plane + (set >> 1 ? (size_t)P.out_W : 0u) + (set & 1u);
      if (P.ksplit > 1u) {
        P.part[((size_t)B.ks * P.num_tiles + pl.tile) * P.part_tile_elems + o] = v;
      } else {
        if (P.beta != 0.f) v += tab[2 * ADH_MAX_TILES + pl.tile][o];
        const_cast<float *>(tab[ADH_MAX_TILES + pl.tile])[o] = v;
      }
    }
  };

  SplitBlock B = next_block(), nB = B;
  uint32_t ch = B.ch_lo, nch;
#pragma unroll
  for (int j = 0; j < XU; ++j) {
    set_unit(B, ch, j);
    load_elems(j, 0, 8);
  }
  load_wrow(B.mg, ch, 0);
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    pack_w(c, 0);
    pack_w(c, 1);
    store_w(c);
  }
  uintx4 b[NT][3], a[2][3];
  bool more = true;
  while (more) {
    lds_barrier();
    store_x();
    lds_barrier();
    const bool last = ch + 1u == B.ch_hi;
    nch = ch + 1u;
    if (last) {
      if (next_vid < end_vid) {
        nB = next_block();
        nch = nB.ch_lo;
      } else {
        more = false;  // (what is prefetched from here on is not used; it reads existing places)
      }
    }
    if (ch == B.ch_lo) {
#pragma unroll
      for (int s = 0; s < SETS; ++s)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int q = 0; q < NT; ++q) acc[s][mt][q] = floatx4{0.f, 0.f, 0.f, 0.f};
      if constexpr (APART) {
#pragma unroll
        for (int s = 0; s < SETS; ++s)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int q = 0; q < NT; ++q) low[s][mt][q] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) a[0][k] = a_lane[k * 4 * kSpMP];
#pragma unroll
    for (int k = 2; k >= 0; --k)
#pragma unroll
      for (int q = 0; q < NT; ++q) b[q][k] = xl[pix[q] + k * 4 * kSpPP];
    static_for<9>([&](auto step) {
      constexpr int t = decltype(step)::value;
      // two steps ahead of the multiplications: tap t2 of this chunk or of the next goes to the slot nobody reads
      constexpr int t2 = (t + 2) % 9, col = t2 % 3, row = t2 / 3;
      uint32_t delta = tap_place((t + 1) / 3, (t + 1) % 3);  // of the next tap
      asm volatile("" : "+s"(delta));  // (the nine taps' addresses are not kept in registers)
      const uintx4 *xb = xl + delta;
      // what follows group i of the step's 6 MT groups of NT multiplications
      auto side = [&](auto group) {
        constexpr int i = decltype(group)::value;
        constexpr int w0 = col == 0 ? 6 * MT - 3 : 0;  // a row's first column late: its loads went out one step ago
        if constexpr (i == w0) pack_w(col, 0);
        if constexpr (i == w0 + 1) pack_w(col, 1);
        if constexpr (i == w0 + 2) {
          store_w(t2 % 3);
          if constexpr (col == 2 && row < 2) load_wrow(B.mg, ch, row + 1);
          if constexpr (col == 2 && row == 2) load_wrow(nB.mg, nch, 0);
        }
        if constexpr (t >= FIRST && t < FIRST + XU) {
          if constexpr (i == 1) set_unit(nB, nch, t - FIRST);
          if constexpr (i % MT == 0 && i / MT >= 1 && i / MT <= 4) {
            if (!idle(t - FIRST)) load_elems(t - FIRST, 2 * (i / MT) - 2, 2 * (i / MT));
          }
        }
      };
      static_for<MT>([&](auto tile) {
        constexpr int mt = decltype(tile)::value, cur = (t * MT + mt) & 1;
        // the next operands: of the next m-tile, or of the next tap's first one
        if constexpr (mt + 1 < MT || t < 8) {
#pragma unroll
          for (int k = 0; k < 3; ++k)
            a[cur ^ 1][k] = mt + 1 < MT ? a_lane[(t % 3) * SLOT + k * 4 * kSpMP + (mt + 1) * 16]
                                        : a_lane[((t + 1) % 3) * SLOT + k * 4 * kSpMP];
        }
        auto &sum = acc[tap_set(t)];
        constexpr bool ONCE = !APART && (LOW == 9 || (t < 2 * LOW && t % 2 == 0));  // this tap's small products are added once
        auto products = [&](auto group, int ka, int kb) {
          constexpr int nth = decltype(group)::value;
#pragma unroll
          for (int q = 0; q < NT; ++q) {
            floatx4 &to = (APART || ONCE) && ka + kb > 0 ? low[APART ? tap_set(t) : 0][APART ? mt : 0][q] : sum[mt][q];
            if (ONCE && nth == 0) to = floatx4{0.f, 0.f, 0.f, 0.f};
            to = VEC ? mfma_bf16(b[q][kb], a[cur][ka], to) : mfma_bf16(a[cur][ka], b[q][kb], to);
          }
          if constexpr (ONCE && nth == 5) {
#pragma unroll
            for (int q = 0; q < NT; ++q) {
              sum[mt][q] += low[0][0][q];
              asm volatile("" : "+v"(sum[mt][q]));  // (stays where it is: moved about, the sums are spilled)
            }
          }
          __builtin_amdgcn_sched_barrier(0);
          side(std::integral_constant<int, mt * 6 + nth>{});
          __builtin_amdgcn_sched_barrier(0);
        };
        auto refill = [&](int kb) {  // the last use of this part of the pixels is behind: fetch the next tap's
          if constexpr (mt + 1 == MT && t < 8) {
#pragma unroll
            for (int q = 0; q < NT; ++q) b[q][kb] = xb[pix[q] + kb * 4 * kSpPP];
          }
        };
        // small products first
        products(std::integral_constant<int, 0>{}, 0, 2);
        refill(2);
        products(std::integral_constant<int, 1>{}, 1, 1);
        products(std::integral_constant<int, 2>{}, 0, 1);
        refill(1);
        products(std::integral_constant<int, 3>{}, 2, 0);
        products(std::integral_constant<int, 4>{}, ONCE ? 0 : 1, 0);  // (the small products' sum is waited for, not h*h's)
        products(std::integral_constant<int, 5>{}, ONCE ? 1 : 0, 0);
        refill(0);
      });
      if (t < 8) lds_barrier();
    });
    if (last) {
      if constexpr (APART) {
#pragma unroll
        for (int s = 0; s < SETS; ++s)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int q = 0; q < NT; ++q) acc[s][mt][q] += low[s][mt][q];
      }
      settle_x();
      if (not_finite == 0u) emit_all(B);
      else emit_plain(B);
      B = nB;
    }
    ch = nch;
  }
}

// out[tile][e] = beta * res[tile][e] + part[0][tile][e] + part[1][tile][e] + ... (a fixed order: reproducible)
__global__ __launch_bounds__(256) void conv3x3_split_reduce_kernel(const SplitParams P) {
  const uint32_t tile = blockIdx.y;
  for (uint64_t e = (uint64_t)blockIdx.x * 256u + threadIdx.x; e < P.part_tile_elems; e += (uint64_t)gridDim.x * 256u) {
    float v = P.part[(size_t)tile * P.part_tile_elems + e];
    for (uint32_t k = 1; k < P.ksplit; ++k) v += P.part[((size_t)k * P.num_tiles + tile) * P.part_tile_elems + e];
    if (P.beta != 0.f) v += P.res[tile][e];
    P.out[tile][e] = v;
  }
}

// ---- host side ----

// How the small products are summed (see LOW), by the relative error against double precision over that of sums of
// v_mfma_f32_16x16x4_f32, for inputs that are uniform in [-1, 1] / normal and rectified.  64 channels: each product by itself 0.83 / 1.12,
// four taps at once 0.68 / 0.91, nine 0.35 / 0.43, apart 0.30 / 0.34; 16 channels, whose chunk has as many additions for half the
// terms: 1.11 / 1.46, 0.93 / 1.23, 0.43 / 0.55, 0.33 / 0.38; one channel, by itself 2.2 / 1.8, apart 0.51 / 0.64.  Backward-data at
// stride 2: 64 channels by itself 0.37 / 0.37, 16 channels 0.96 / 0.98, three 1.95 / 1.47.
// 64 -> 64 channels on 32 x 128 tiles (32 images, 4 tiles): by itself 215 us, four taps 215, nine 235, apart (half the tile, for the
// registers) 260.
static int split_low(SplitSample sample, uint32_t C, uint32_t nchunks) {
  if (sample == kDown) return kLowApart;  // (one set of sums, and the registers for two)
  if (sample == kUp) return C < 16u ? kLowApart : 0;
  return C <= 4u ? kLowApart : 8u * C >= 7u * kSpChunk * nchunks ? 4 : 9;
}

struct SplitPlan {
  SplitParams P;
  int MT, NT, low;
  bool vec;
  double cycles;  // expected
  size_t part_bytes;
};

// Blocks of BR x BC output pixels (of NB images) by 16 MT channels.  The workgroups are persistent, one per compute unit, so
// a launch takes ceil(blocks / 256) times a block.  A block's cycles, as measured in the kernel: nine steps a chunk, each a
// SIMD's 2 * 6 * 16 * MT * NT matrix cycles (at least 1300: its barrier, staging and operand reads) and 300 more; 1500 and
// 2000 NT a chunk for loading, splitting and changing the patch; the results.  Where that leaves compute units idle and there
// is a workspace, a block's chunks are dealt to several workgroups and a second kernel adds their sums, at its launch and the
// sums' way through memory (1.2 KB a cycle): 512 channels on 4 tiles of 2 x 8, 32 images, 130 -> 74 us; on one image of 14 x 14
// a tile 124 -> 40; 256 -> 512 on 28 x 28, 8 images, backward-data 147 -> 95.
// The choice is made anew on every call, so tiles that cannot win are passed over by their least number of blocks before they are
// priced: 64 channels on 4 x 32 x 128 5.8 -> 1.2 us of host time, on 8 x 128 x 2048 10.8 -> 1.6, the median of random shapes
// 3.9 -> 1.5, with the same choices.
static double split_chunk_cycles(int MT, int NT) { return 9.0 * (std::max(192.0 * MT * NT, 1300.0) + 300.0) + 1500.0 + 2000.0 * NT; }
static double split_results_cycles(SplitSample sample, int MT, int NT) { return 2000.0 + 500.0 * MT * NT * (sample == kUp ? 4 : 1); }
constexpr double kSplitDealtCycles = 9000.0;  // the second kernel's launch

static int split_plan(const Conv3x3Problem &q, bool workspace, SplitPlan *plan) {
  SplitParams &P = plan->P;
  P.N = q.N; P.C = q.C; P.M = q.M; P.num_tiles = q.num_tiles;
  P.NI = q.stacked ? q.N : q.N * q.num_tiles;
  P.in_H = q.in_H; P.in_W = q.in_W; P.out_H = q.out_H; P.out_W = q.out_W;
  P.in_VH = q.in_H; P.grid_VH = q.out_H; P.grid_W = q.sample == kUp ? q.in_W : q.out_W;
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
  P.nchunks = (P.C + kSpChunk - 1u) / kSpChunk;
  plan->low = split_low(q.sample, P.C, P.nchunks);
  const double out_bytes = 4.0 * P.num_tiles * P.N * P.M * P.out_H * P.out_W;
  const uint32_t pixels = split_patch(q.sample);
  // extent of the patch of n pixels, and how many pixels one of n holds
  auto patch = [&](uint32_t n) { return q.sample == kDown ? 2u * n + 1u : q.sample == kUp ? n + 1u : n + 2u * q.dil; };
  auto held = [&](uint32_t n) { return n < patch(1u) ? 0u : q.sample == kDown ? (n - 1u) / 2u : n - (patch(1u) - 1u); };
  double best = 1e300;
  uint32_t nbi = 0, nbj = 0;
  const uint64_t grid_rows = (uint64_t)P.NI * P.grid_VH, grid_pixels = grid_rows * P.grid_W;
  for (int MT = P.M <= 16u ? 1 : P.M <= 32u ? 2 : 4; MT >= 1; MT /= 2) {
    const uint32_t MG = (P.M + 16u * MT - 1u) / (16u * MT);
    for (int NT = q.sample == kDown ? 1 : 4; NT >= 1; NT /= 2) {
      if (q.sample == kUp && NT == 4 && MT > 1) continue;  // (four sets of sums)
      // (what the registers hold of two sets of sums: at stride 1 the largest such tile of each height)
      if (plan->low == kLowApart && (q.sample == kUnit ? NT != (MT == 1 ? 4 : 2) : q.sample == kUp && NT > 1 && MT * NT > 2)) continue;
      const uint32_t slots = 128u * NT;
      const double chunk = split_chunk_cycles(MT, NT), results = split_results_cycles(q.sample, MT, NT);
      // What `blocks` blocks cost, their chunks undealt or (where they leave compute units idle) as dealt at best.  It grows with
      // their number, so that tiles whose least possible number costs more than the best plan so far are passed over.
      auto undealt = [&](uint64_t blocks) { return (double)((blocks + 255u) / 256u) * (P.nchunks * chunk + results) + 1e-3 * (double)blocks; };
      auto dealt = [&](uint64_t blocks, uint32_t cps, uint32_t ks) {
        return cps * chunk + results + kSplitDealtCycles + out_bytes * (ks + 1) / 1200.0 + 1e-3 * (double)blocks;
      };
      auto worse = [&](uint64_t least) {
        if (undealt(least) < best) return false;
        const uint64_t most = workspace ? 256u / least : 1u;
        return most < 2u || dealt(least, (uint32_t)((P.nchunks + most - 1u) / most), 2u) >= best;
      };
      if (worse((grid_pixels + slots - 1u) / slots * MG)) continue;
      // columns per block: whole rows, halves and so on down to eight, multiples of four where rows are
      for (uint32_t parts = (P.grid_W + 255u) / 256u; parts <= P.grid_W; parts += 1u + parts / 8u) {
        uint32_t BC = (P.grid_W + parts - 1u) / parts;
        if (parts > 1u && BC < 8u) break;
        if (P.grid_W % 4u == 0u) BC = (BC + 3u) & ~3u;
        if (BC > slots) continue;
        const uint32_t nc = (P.grid_W + BC - 1u) / BC, rows = slots / BC;
        if (worse((grid_rows + rows - 1u) / rows * nc * MG)) continue;
        const uint32_t patch_BC = patch(BC), max_BR = std::min(std::min(P.grid_VH, rows), held(pixels / patch_BC));
        if (max_BR == 0u) continue;
        const uint32_t nr0 = (P.grid_VH + max_BR - 1u) / max_BR;
        for (uint32_t nr = nr0; nr < nr0 + 2u && nr <= P.grid_VH; ++nr) {
          const uint32_t BR = (P.grid_VH + nr - 1u) / nr;
          uint32_t NB = std::min(std::min(rows / BR, pixels / (patch(BR) * patch_BC)), P.NI);
          const uint32_t groups = (P.NI + NB - 1u) / NB;
          const uint64_t blocks = (uint64_t)groups * nc * nr * MG;
          auto keep = [&](double cost, uint32_t ks, uint32_t cps) {
            if (cost >= best) return;
            best = cost;
            plan->MT = MT; plan->NT = NT;
            P.BR = BR; P.BC = BC; P.NB = (P.NI + groups - 1u) / groups;
            P.ksplit = ks; P.chunks_per_split = cps;
            nbi = nr; nbj = nc;
          };
          keep(undealt(blocks), 1u, P.nchunks);
          // chunks dealt to several workgroups per block, while all of them run at once
          const uint64_t most = workspace ? 256u / blocks : 1u;
          if (most < 2u) continue;
          uint32_t ks = 1;
          for (uint32_t cps = P.nchunks - 1u; cps >= 1u; --cps) {
            ks = (P.nchunks + cps - 1u) / cps;
            if (ks > most) break;
            keep(dealt(blocks, cps, ks), ks, cps);
          }
        }
      }
    }
  }
  if (nbi == 0u) return ADH_EUNIMPL;
  plan->cycles = best;
  const uint32_t MG = (P.M + 16u * plan->MT - 1u) / (16u * plan->MT), PCP = patch(P.BC), PPI = patch(P.BR) * PCP;
  P.PPn = P.NB * PPI;
  plan->vec = P.BC % 4u == 0u && P.grid_W % 4u == 0u;
  const uint64_t base = (uint64_t)((P.NI + P.NB - 1u) / P.NB) * nbi * nbj * MG;
  if (base * P.ksplit >= (1ull << 30)) return ADH_EUNIMPL;
  P.blocks = (uint32_t)(base * P.ksplit);
  P.xcd_chunk = (P.blocks + 7u) / 8u;
  P.part_tile_elems = (uint64_t)P.N * P.M * P.out_H * P.out_W;
  plan->part_bytes = P.ksplit > 1u ? (size_t)P.ksplit * P.num_tiles * P.part_tile_elems * 4u : 0u;
  P.div_bpg = FastDiv(nbi * nbj); P.div_nbj = FastDiv(nbj); P.div_MG = FastDiv(MG); P.div_N = FastDiv(P.N);
  P.div_BC = FastDiv(P.BC); P.div_live = FastDiv(P.BR * P.BC); P.div_PPI = FastDiv(PPI); P.div_PCP = FastDiv(PCP);
  P.div_PPn = FastDiv(P.PPn); P.div_ksplit = FastDiv(P.ksplit); P.div_in = FastDiv(P.in_step); P.div_out = FastDiv(P.out_step);
  return ADH_OK;
}

size_t conv3x3_split_workspace(const Conv3x3Problem &q) {
  SplitPlan plan = {};
  return split_plan(q, true, &plan) ? 0u : (plan.part_bytes + 255u) & ~(size_t)255u;
}

constexpr double kSplitCyclesPerUs = 2100.0;
// No plan is expected to take less than a block of the smallest tile, of all chunks or (with a workspace) of one of them: what tells
// small launches, which go to conv_f32_patch.hip, without a plan.
static double split_least_us(const Conv3x3Problem &q, bool workspace) {
  const uint32_t nchunks = (q.C + kSpChunk - 1u) / kSpChunk;
  const double chunk = split_chunk_cycles(1, 1), results = split_results_cycles(q.sample, 1, 1), whole = nchunks * chunk + results;
  return (workspace ? std::min(whole, chunk + results + kSplitDealtCycles) : whole) / kSplitCyclesPerUs;
}

bool conv3x3_split_exceeds(const Conv3x3Problem &q, bool workspace, double most_us) {
  if (split_least_us(q, workspace) > most_us) return true;
  SplitPlan plan = {};
  return split_plan(q, workspace, &plan) || plan.cycles / kSplitCyclesPerUs > most_us;
}

bool conv3x3_split_idles(const Conv3x3Problem &q) {
  SplitPlan plan = {};
  if (split_plan(q, false, &plan)) return false;
  const uint32_t rounds = (plan.P.blocks + 255u) / 256u;
  return rounds > 1u && (rounds * 256u - plan.P.blocks) * 8u > rounds * 256u;
}

void conv3x3_split_name(const Conv3x3Problem &q, char *name, size_t name_bytes) {
  SplitPlan plan = {};
  if (split_plan(q, false, &plan)) plan.MT = plan.NT = 0;
  snprintf(name, name_bytes, "conv3x3_split_kernel<%d, %d, %s, %d, %d>", plan.MT, plan.NT, plan.vec ? "true" : "false", (int)q.sample, plan.low);
}

template <int MT, int NT, int SAMPLE, int LOW>
static void launch_split(const SplitPlan &plan, hipStream_t st) {
  const dim3 grid(std::min(plan.P.xcd_chunk, 32u) * 8u), block(kSpThreads);
  if (plan.vec) hipLaunchKernelGGL((conv3x3_split_kernel<MT, NT, true, SAMPLE, LOW>), grid, block, 0, st, plan.P);
  else hipLaunchKernelGGL((conv3x3_split_kernel<MT, NT, false, SAMPLE, LOW>), grid, block, 0, st, plan.P);
}
template <int MT>
static void launch_split_nt(const SplitPlan &plan, SplitSample sample, hipStream_t st) {
  const bool apart = plan.low == kLowApart;
  if (sample == kDown) {
    launch_split<MT, 1, kDown, kLowApart>(plan, st);
  } else if (sample == kUp) {
    if (MT == 1 && plan.NT == 4) launch_split<1, 4, kUp, 0>(plan, st);
    else if (plan.NT == 2) apart ? launch_split<1, 2, kUp, kLowApart>(plan, st) : launch_split<MT, 2, kUp, 0>(plan, st);
    else apart ? launch_split<MT, 1, kUp, kLowApart>(plan, st) : launch_split<MT, 1, kUp, 0>(plan, st);
  } else if (apart) {
    launch_split<MT, MT == 1 ? 4 : 2, kUnit, kLowApart>(plan, st);
  } else if (plan.NT == 4) {
    plan.low == 4 ? launch_split<MT, 4, kUnit, 4>(plan, st) : launch_split<MT, 4, kUnit, 9>(plan, st);
  } else if (plan.NT == 2) {
    plan.low == 4 ? launch_split<MT, 2, kUnit, 4>(plan, st) : launch_split<MT, 2, kUnit, 9>(plan, st);
  } else {
    plan.low == 4 ? launch_split<MT, 1, kUnit, 4>(plan, st) : launch_split<MT, 1, kUnit, 9>(plan, st);
  }
}

int conv3x3_split(const Conv3x3Problem &q, void *workspace, size_t workspace_bytes, double most_us, hipStream_t st) {
  if (split_least_us(q, workspace != nullptr) > most_us) return ADH_EUNIMPL;
  SplitPlan plan = {};
  int e = split_plan(q, workspace != nullptr, &plan);
  if (e == ADH_OK && plan.cycles / kSplitCyclesPerUs > most_us) return ADH_EUNIMPL;
  if (e == ADH_OK && plan.part_bytes > workspace_bytes) {
    plan = {};
    e = split_plan(q, false, &plan);
  }
  if (e) return e;
  SplitParams &P = plan.P;
  for (uint32_t t = 0; t < q.num_tiles; ++t) {
    P.in[t] = reinterpret_cast<const float *>(q.in[t]);
    P.out[t] = reinterpret_cast<float *>(q.out[t]);
    P.res[t] = reinterpret_cast<const float *>(q.res ? q.res[t] : q.out[t]);
  }
  P.w = reinterpret_cast<const float *>(q.w);
  P.part = reinterpret_cast<float *>(workspace);
  if (plan.MT == 4) launch_split_nt<4>(plan, q.sample, st);
  else if (plan.MT == 2) launch_split_nt<2>(plan, q.sample, st);
  else launch_split_nt<1>(plan, q.sample, st);
  if (P.ksplit > 1u) {
    const uint32_t rb = (uint32_t)std::min<uint64_t>((P.part_tile_elems + 255u) / 256u, 2048u);
    hipLaunchKernelGGL(conv3x3_split_reduce_kernel, dim3(rb, q.num_tiles), dim3(256), 0, st, P);
  }
  return launch_status();
}

}  // namespace adh
