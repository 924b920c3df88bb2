// Filter gradient of the 3x3 window at stride 1 in fp32 on the bf16 matrix cores (split_bf16.h says how):
//   dw[co][ci][a][b] = beta*dw + sum over images, R, Q of dy[co][R][Q] * x[ci][R + a - pad_r][Q + b - pad_c]
//
// Mapping.  Per tap D[co][ci] += A[co][pixel] B[pixel][ci] on v_mfma_f32_16x16x32_bf16, k = 32 pixels: four octets of
// neighbouring pixels of a row.  Both tensors lie in LDS as [row][octet][channel] (octet_swap), in three parts; an operand is one
// ds_read_b128, and the window's second and third columns come from the same octet and the next one's first columns (a
// ds_read_b64: 4.3 cycles, a dword 8) by v_alignbit.
//   * A workgroup of eight waves, one per compute unit, owns 32*OT output channels x 32*CT input channels x nine taps and a
//     run of steps; a step is RS rows of TW columns (2 x 32, 4 x 16 or 8 x 8), half of its octets for each half of the
//     waves.  A wave keeps 16*OT x 16*CT x 9 sums: at OT = CT = 2 a step is 216 MFMAs
//     a wave (3456 matrix cycles) against 42 operand reads and 144 shifts.
//   * x rows go through a ring of 2 RS + 2 rows and dy rows through two buffers: a step brings RS new rows of each.  The rows
//     of the next step are split and stored while this one is multiplied, and the ones after those are on their way in
//     registers; the two waves of a SIMD take turns, one staging while the other multiplies.  One barrier a step.
//   * What is multiplied need not be there: a step may reach past dy's last column or row, where dy is zero and x is whatever lies
//     beside it, and an infinity's parts are not all finite.  Either way (zero times a NaN, inf - inf) the sum comes out as NaN:
//     sums that are NaN are computed over again in plain fp32 from the pixels that exist.  (Noting such values as they are
//     staged takes instructions and registers in the loop.)
//   * The halves' sums are added through LDS, the workgroups' by a second kernel in a fixed order (reproducible).
// Row tiles of one tensor are addressed as that tensor (as in conv3x3_split.hip).
//
// Measured (32 images, 4 tiles without halo; the v_mfma_f32 kernel before): 64 channels on 32 x 128 tiles 0.351 -> 0.197 ms
// (196 TFLOP/s), 128 on 16 x 64 0.354 -> 0.193, 256 on 8 x 32 0.361 -> 0.195, 512 on 4 x 16 0.456 -> 0.21 (0.61 through the
// general entry point before); with [octet][channel] rows in place of [channel][pixel] ones, where bank conflicts took 0.41 of all cycles,
// 0.181, 0.173, 0.175, 0.192, and 1.08 times as fast in the mean of 115 layers (176 -> 16 channels on 3 tiles of 7 x 391 116 -> 91 us); with what a step's loads need read where it is used (from_memory), 0.989 of the
// time over 60 random padded layers.  Staging: with rows, channels and tiles worked out per group of four values the kernel took
// 0.45 ms; a thread's channel and column fixed and a wave's row uniform it is a load, a split and three writes.  Bound: a
// step of 6912 matrix cycles takes about 11000, the splitting and the shifts (a third of the issue slots) and the clock,
// which the power limit holds at 1.8 - 2.1 GHz; and on short layers the workgroups' sums, 38 MB written and read back.
#include "conv3x3_wgrad_split.h"

#include <algorithm>

#include "split_bf16.h"

namespace adh {

constexpr uint32_t kWsThreads = 512;
constexpr uint32_t kWsLdsBytes = 163072;

struct WgradSplitParams {
  const float *x[ADH_MAX_TILES], *dy[ADH_MAX_TILES];
  float *part;  // [channel group][split][wave tile][ot][ct][tap][lane][4]
  float *dw;
  uint32_t N, Cin, Cout, num_tiles;
  uint32_t x_H, x_W, dy_H, dy_W, x_VH, dy_VH, step, last_tile;
  int32_t pad_r, pad_c, neighbours;
  uint32_t TW, logQ, RS, NR;                // logQ: log2 of a row's groups of four columns
  uint32_t x_row_bytes, dy_row_bytes;       // of one part of a row of x (with the octet behind it) and of dy
  uint32_t x_part_bytes, dy_part_bytes;     // bytes of one part of the ring and of the dy buffers
  uint32_t col_tiles, row_steps, total_steps, splits, ci_groups, group0;
  float beta;
  FastDiv div_row_steps, div_cols, div_N, div_step, div_splits, div_cig;
};

template <int OT, int CT>
__global__ __launch_bounds__(kWsThreads, 2) void conv3x3_wgrad_split_kernel(const WgradSplitParams args) {
  const WgradSplitParams &P = args;
  constexpr uint32_t CO = 32u * OT, CI = 32u * CT;
  __shared__ __align__(16) char lds[kWsLdsBytes];
  __shared__ uint32_t nan_sums;
  char *const dyl = lds + 3u * P.x_part_bytes;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t half = wave >> 2, wo = wave & 1u, wc = (wave >> 1) & 1u;

  uint32_t group, split, cog, cig;
  P.div_splits.divmod(blockIdx.x, group, split);
  P.div_cig.divmod(P.group0 + group, cog, cig);
  const uint32_t co0 = cog * CO, ci0 = cig * CI;
  uint32_t s = (uint32_t)((uint64_t)P.total_steps * split / P.splits);
  const uint32_t s_end = (uint32_t)((uint64_t)P.total_steps * (split + 1u) / P.splits);

  if (tid == 0u) nan_sums = 0u;
  lds_barrier();

  // the run that the workgroup stands in: an image (pair) and a column tile of it
  uint32_t tile0 = 0, n = 0, c0 = 0;
  const size_t x_plane = (size_t)P.x_H * P.x_W, dy_plane = (size_t)P.dy_H * P.dy_W;
  // tile and row of the stacked tensor's row R; of x row R where the halo rows are the neighbours' interior rows
  struct Row { uint32_t tile, r; };
  auto row_of = [&](const WgradSplitParams &P, uint32_t R, bool is_x) {
    const uint32_t t = min(P.div_step.div(R), P.last_tile);
    Row w = {tile0 + t, R - t * P.step};
    if (P.neighbours && is_x) {
      if (R == 0u && tile0 > 0u) w = {tile0 - 1u, P.dy_H};
      else if (R == P.dy_H + 1u && tile0 + 1u < P.num_tiles) w = {tile0 + 1u, 1u};
    }
    return w;
  };

  // Staging.  A step's rows of TW = 4 << logQ columns are 1024 groups of four columns per 64 channels: a thread takes one of
  // every 512, whose channel and column are the same for all of them and whose row is the same for the whole wave.  Of the
  // two x columns more that the window's last columns want, a wave takes one row, a lane one channel.
  const uint32_t q = tid & ((1u << P.logQ) - 1u), c_x = (tid >> P.logQ) & (CI - 1u), c_dy = (tid >> P.logQ) & (CO - 1u);
  const uint32_t x_rows = kWsThreads / (CI << P.logQ), dy_rows = kWsThreads / (CO << P.logQ);  // per 512 groups
  const uint32_t x_row = (wave * 64u) >> P.logQ >> (CT == 2 ? 6 : 5), dy_row = (wave * 64u) >> P.logQ >> (OT == 2 ? 6 : 5);
  const bool c_x_ok = ci0 + c_x < P.Cin, c_dy_ok = co0 + c_dy < P.Cout, c_tail_ok = lane < CI && ci0 + lane < P.Cin;
  const uint32_t x_to = ((q >> 1) * CI + (c_x ^ octet_swap(q >> 1))) * 16u + (q & 1u) * 8u, dy_to = ((q >> 1) * CO + (c_dy ^ octet_swap(q >> 1))) * 16u + (q & 1u) * 8u;
  const size_t x_chan = (size_t)(c_x_ok ? ci0 + c_x : 0u) * x_plane, dy_chan = (size_t)(c_dy_ok ? co0 + c_dy : 0u) * dy_plane;
  const size_t tail_chan = (size_t)(c_tail_ok ? ci0 + lane : 0u) * x_plane;
  // columns by which four loaded values lie left of the wanted ones (they are loaded inside the row); 4: none exists
  int32_t x_from = 0, x_shift = 0, dy_from = 0, dy_shift = 0;
  auto place = [](int32_t Q, int32_t W, bool ok, int32_t &from, int32_t &shift) {
    from = min(max(Q, 0), max(W - 4, 0));
    shift = ok && Q > -4 && Q < W ? Q - from : 4;
  };
  constexpr int XR = CT, DR = OT;  // groups of four a thread stages per step
  floatx4 vx[XR], vd[DR];
  float tail[2];
  const int32_t xW = (int32_t)P.x_W, dW = (int32_t)P.dy_W;
  auto load4 = [&](const float *row, int32_t from, int32_t W) {
    const ADH_GLOBAL float *p = (const ADH_GLOBAL float *)row + from;
    if (W >= 4) return *(const ADH_GLOBAL floatx4_u *)p;
    const float a = p[0], b = W > 1 ? p[1] : 0.f, c = W > 2 ? p[2] : 0.f;
    return floatx4_u{a, b, c, 0.f};
  };
  // x rows x0 .. x0 + nx - 1 (of the padded numbering), dy rows d0 .. d0 + nd - 1
  auto load = [&](uint32_t x0, uint32_t nx, uint32_t d0, uint32_t nd) {
    const WgradSplitParams &P = from_memory(args);
#pragma unroll
    for (int j = 0; j < XR; ++j) {
      const uint32_t i = (uint32_t)j * x_rows + x_row;
      const int32_t R = (int32_t)(x0 + i) - P.pad_r;
      if (i < nx && R >= 0 && R < (int32_t)P.x_VH) {
        const Row w = row_of(P, (uint32_t)R, true);
        vx[j] = load4(P.x[w.tile] + ((size_t)n * P.Cin * x_plane + (size_t)w.r * P.x_W) + x_chan, x_from, xW);
      } else {
        vx[j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int j = 0; j < DR; ++j) {
      const uint32_t i = (uint32_t)j * dy_rows + dy_row, R = d0 + i;
      if (i < nd && R < P.dy_VH) {
        const Row w = row_of(P, R, false);
        vd[j] = load4(P.dy[w.tile] + ((size_t)n * P.Cout * dy_plane + (size_t)w.r * P.dy_W) + dy_chan, dy_from, dW);
      } else {
        vd[j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
    }
    const int32_t R = (int32_t)(x0 + wave) - P.pad_r, Q = (int32_t)(c0 + P.TW) - P.pad_c;
    tail[0] = tail[1] = 0.f;
    if (wave < nx && R >= 0 && R < (int32_t)P.x_VH) {
      const Row w = row_of(P, (uint32_t)R, true);
      const ADH_GLOBAL float *p = (const ADH_GLOBAL float *)P.x[w.tile] + ((size_t)n * P.Cin * x_plane + (size_t)w.r * P.x_W) + tail_chan;
      if (Q < xW) tail[0] = p[Q];
      if (Q + 1 < xW) tail[1] = p[Q + 1];
    }
  };
  auto moved = [](floatx4 y, int32_t d) {
    if (__builtin_amdgcn_ballot_w64(d != 0)) {
#pragma unroll
      for (int k = 1; k < 4; ++k) {  // columns before the row's first one
        const bool move = d <= -k;
        y = floatx4{move ? 0.f : y[0], move ? y[0] : y[1], move ? y[1] : y[2], move ? y[2] : y[3]};
      }
#pragma unroll
      for (int k = 1; k < 4; ++k) {  // columns past its last one
        const bool move = d >= k;
        y = floatx4{move ? y[1] : y[0], move ? y[2] : y[1], move ? y[3] : y[2], move ? 0.f : y[3]};
      }
      const bool none = d >= 4;
      y = floatx4{none ? 0.f : y[0], none ? 0.f : y[1], none ? 0.f : y[2], none ? 0.f : y[3]};
    }
    return y;
  };
  // slot0: ring slot of x row x0; buf: the dy buffer
  auto store = [&](uint32_t slot0, uint32_t nx, uint32_t buf, uint32_t nd) {
    auto put = [&](floatx4 y, char *p, uint32_t stride) {
      uint32_t part[3][2];
      split_pair(y[0], y[1], part[0][0], part[1][0], part[2][0]);
      split_pair(y[2], y[3], part[0][1], part[1][1], part[2][1]);
#pragma unroll
      for (int k = 0; k < 3; ++k) *reinterpret_cast<uintx2 *>(p + k * stride) = uintx2{part[k][0], part[k][1]};
    };
    auto slot_of = [&](uint32_t i) {
      const uint32_t slot = slot0 + i;
      return slot - (slot >= P.NR ? P.NR : 0u);
    };
#pragma unroll
    for (int j = 0; j < XR; ++j) {
      const uint32_t i = (uint32_t)j * x_rows + x_row;
      if (i < nx) put(moved(vx[j], x_shift), lds + slot_of(i) * P.x_row_bytes + x_to, P.x_part_bytes);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < DR; ++j) {
      const uint32_t i = (uint32_t)j * dy_rows + dy_row;
      if (i < nd) put(moved(vd[j], dy_shift), dyl + (buf * P.RS + i) * P.dy_row_bytes + dy_to, P.dy_part_bytes);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (wave < nx && lane < CI) {
      if (!c_tail_ok) tail[0] = tail[1] = 0.f;
      uint32_t part[3];
      split_pair(tail[0], tail[1], part[0], part[1], part[2]);
      char *p = lds + slot_of(wave) * P.x_row_bytes + ((P.TW >> 3) * CI + (lane ^ octet_swap(P.TW >> 3))) * 16u;
#pragma unroll
      for (int k = 0; k < 3; ++k) *reinterpret_cast<uint32_t *>(p + k * P.x_part_bytes) = part[k];
    }
  };

  // ---- this lane group's octet of a step: row io of the step, octet qo of the row ----
  const uint32_t oct = half * 4u + g, io = oct >> (P.logQ - 1u), qo = oct & ((1u << (P.logQ - 1u)) - 1u);
  const uint32_t b_base = (qo * CI + wc * CT * 16u + (l16 ^ octet_swap(qo))) * 16u, e_base = ((qo + 1u) * CI + wc * CT * 16u + (l16 ^ octet_swap(qo + 1u))) * 16u;
  const uint32_t a_base = io * P.dy_row_bytes + (qo * CO + wo * OT * 16u + (l16 ^ octet_swap(qo))) * 16u;

  floatx4 acc[OT][CT][9];
#pragma unroll
  for (int ot = 0; ot < OT; ++ot)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int t = 0; t < 9; ++t) acc[ot][ct][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  // base: ring slot of the step's first x row
  auto multiply = [&](uint32_t base, uint32_t buf) {
    uintx4 a[OT][3];
#pragma unroll
    for (int ot = 0; ot < OT; ++ot)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        a[ot][k] = *reinterpret_cast<const uintx4 *>(dyl + k * P.dy_part_bytes + a_base + ot * 256u + buf * P.RS * P.dy_row_bytes);
    struct Operand { uintx4 d; uintx2 e; };  // an octet, the next one's first columns
    Operand b[2][3];
    auto fetch = [&](int set, int r, int ct) {
      uint32_t slot = base + io + (uint32_t)r;
      slot -= slot >= P.NR ? P.NR : 0u;
      const char *p = lds + slot * P.x_row_bytes + ct * 256u;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        b[set][k].d = *reinterpret_cast<const uintx4 *>(p + b_base + k * P.x_part_bytes);
        b[set][k].e = *reinterpret_cast<const uintx2 *>(p + e_base + k * P.x_part_bytes);
      }
    };
    fetch(0, 0, 0);
#pragma unroll
    for (int i = 0; i < 3 * CT; ++i) {
      const int r = i / CT, ct = i % CT, cur = i & 1;
      if (i + 1 < 3 * CT) fetch(cur ^ 1, (i + 1) / CT, (i + 1) % CT);
      uintx4 w[3][3];  // part, window column
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        uintx4 d = b[cur][k].d;
        asm("" : "+v"(d));  // (the compiler would read the shifted columns from LDS again, dword by dword)
        const uint32_t e = b[cur][k].e[0];
        w[k][0] = d;
        w[k][1] = uintx4{__builtin_amdgcn_alignbit(d[1], d[0], 16), __builtin_amdgcn_alignbit(d[2], d[1], 16),
                         __builtin_amdgcn_alignbit(d[3], d[2], 16), __builtin_amdgcn_alignbit(e, d[3], 16)};
        w[k][2] = uintx4{d[1], d[2], d[3], e};
      }
      auto products = [&](int ka, int kb) {
#pragma unroll
        for (int col = 0; col < 3; ++col)
#pragma unroll
          for (int ot = 0; ot < OT; ++ot) acc[ot][ct][r * 3 + col] = mfma_bf16(a[ot][ka], w[kb][col], acc[ot][ct][r * 3 + col]);
      };
      // small products first
      products(0, 2); products(1, 1); products(2, 0); products(0, 1); products(1, 0); products(0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  while (s < s_end) {
    // a run: steps of one image (pair) and column tile
    const WgradSplitParams &M = from_memory(args);
    uint32_t run, rs, img, ctile;
    M.div_row_steps.divmod(s, run, rs);
    M.div_cols.divmod(run, img, ctile);
    M.div_N.divmod(img, tile0, n);
    c0 = ctile * P.TW;
    const uint32_t steps = min(s_end - s, M.row_steps - rs);
    place((int32_t)(c0 + 4u * q) - P.pad_c, xW, c_x_ok, x_from, x_shift);
    place((int32_t)(c0 + 4u * q), dW, c_dy_ok, dy_from, dy_shift);
    uint32_t r0 = rs * P.RS, base = 0, buf = 0;
    load(r0, 2u, 0u, 0u);
    lds_barrier();  // every wave is done with the run before
    store(0u, 2u, 0u, 0u);
    load(r0 + 2u, P.RS, r0, P.RS);
    store(2u, P.RS, 0u, P.RS);
    if (steps > 1u) load(r0 + P.RS + 2u, P.RS, r0 + P.RS, P.RS);
    lds_barrier();
    for (uint32_t k = 0; k < steps; ++k) {
      auto stage = [&]() {
        if (k + 1u < steps) {
          uint32_t slot = base + P.RS + 2u;
          slot -= slot >= P.NR ? P.NR : 0u;
          store(slot, P.RS, buf ^ 1u, P.RS);
          if (k + 2u < steps) load(r0 + 2u * P.RS + 2u, P.RS, r0 + 2u * P.RS, P.RS);
        }
      };
      // the two waves of a SIMD take turns: one stages while the other multiplies
      if (half == 0u) stage();
      __builtin_amdgcn_sched_barrier(0);
      multiply(base, buf);
      __builtin_amdgcn_sched_barrier(0);
      if (half != 0u) stage();
      r0 += P.RS;
      base += P.RS;
      base -= base >= P.NR ? P.NR : 0u;
      buf ^= 1u;
      if (k + 1u < steps) lds_barrier();
    }
    s += steps;
  }

  // ---- the halves' sums, then to the workspace ----
  lds_barrier();
  constexpr uint32_t kTile = 9u * 256u;
  floatx4 *const other = reinterpret_cast<floatx4 *>(lds) + (wave & 3u) * (OT * CT * 9u * 64u) + lane;
  if (half != 0u) {
#pragma unroll
    for (int ot = 0; ot < OT; ++ot)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int t = 0; t < 9; ++t) other[((ot * CT + ct) * 9 + t) * 64] = acc[ot][ct][t];
  }
  lds_barrier();
  float *const part = P.part + (size_t)blockIdx.x * (4u * OT * CT * kTile);
  if (half == 0u) {
    ADH_GLOBAL float *out = (ADH_GLOBAL float *)part + (size_t)wave * (OT * CT * kTile) + lane * 4u;
    bool nan = false;
#pragma unroll
    for (int ot = 0; ot < OT; ++ot)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          const floatx4 sum = acc[ot][ct][t] + other[((ot * CT + ct) * 9 + t) * 64];
          nan |= __builtin_isunordered(sum[0], sum[1]) || __builtin_isunordered(sum[2], sum[3]);
          *(ADH_GLOBAL floatx4_u *)(out + ((ot * CT + ct) * 9 + t) * 256) = sum;
        }
    if (nan) nan_sums = 1u;
  }
  __syncthreads();
  if (nan_sums == 0u) return;
  // sums that are NaN once more in plain fp32, straight from memory
  const WgradSplitParams &M = from_memory(args);
  s = (uint32_t)((uint64_t)M.total_steps * split / M.splits);
  for (uint32_t at = tid; at < 4u * OT * CT * kTile; at += kWsThreads) {
    if (part[at] == part[at]) continue;
    const uint32_t i = at & 3u, ln = at >> 2 & 63u, rest = at >> 8, tap = rest % 9u, ct = rest / 9u % CT, ot = rest / 9u / CT % OT;
    const uint32_t wt = rest / 9u / CT / OT;
    const uint32_t co = co0 + ((wt & 1u) * OT + ot) * 16u + (ln >> 4) * 4u + i, ci = ci0 + ((wt >> 1) * CT + ct) * 16u + (ln & 15u);
    float sum = 0.f;
    if (co < M.Cout && ci < M.Cin)
      for (uint32_t st = s; st < s_end && sum == sum; ++st) {  // (a NaN stays one)
        uint32_t run, rs, img, ctile;
        M.div_row_steps.divmod(st, run, rs);
        M.div_cols.divmod(run, img, ctile);
        M.div_N.divmod(img, tile0, n);
        for (uint32_t R = rs * M.RS; R < min((rs + 1u) * M.RS, M.dy_VH) && sum == sum; ++R)
          for (uint32_t Q = ctile * M.TW; Q < min((ctile + 1u) * M.TW, M.dy_W) && sum == sum; ++Q) {
            const int32_t xr = (int32_t)(R + tap / 3u) - M.pad_r, xc = (int32_t)(Q + tap % 3u) - M.pad_c;
            float xe = 0.f;
            if (xr >= 0 && xr < (int32_t)M.x_VH && xc >= 0 && xc < (int32_t)M.x_W) {
              const Row w = row_of(M, (uint32_t)xr, true);
              xe = M.x[w.tile][((size_t)n * M.Cin + ci) * x_plane + (size_t)w.r * M.x_W + (uint32_t)xc];
            }
            const Row w = row_of(M, R, false);
            sum = __builtin_fmaf(M.dy[w.tile][((size_t)n * M.Cout + co) * dy_plane + (size_t)w.r * M.dy_W + Q], xe, sum);
          }
      }
    part[at] = sum;
  }
}

// dw = beta*dw + the splits' sums.  Sixteen lanes take sixteen neighbouring groups of four sums and 16 slices of the splits
// each (slice j: splits j, j + 16, ..); the slices are then added in order: a fixed order, so the result has fixed bits.
template <int OT, int CT>
__global__ __launch_bounds__(256) void conv3x3_wgrad_split_reduce_kernel(const WgradSplitParams P) {
  __shared__ floatx4 sums[16][16];
  constexpr uint32_t kQuads = 4u * OT * CT * 9u * 64u;  // of a channel group
  const uint32_t quad = blockIdx.x * 16u + (threadIdx.x & 15u), slice = threadIdx.x >> 4;
  const uint32_t group = quad / kQuads, e = quad - group * kQuads;
  const floatx4 *p = reinterpret_cast<const floatx4 *>(P.part) + (size_t)group * P.splits * kQuads + e;
  floatx4 sum = {0.f, 0.f, 0.f, 0.f};
  for (uint32_t k = slice; k < P.splits; k += 16u) sum += *reinterpret_cast<const floatx4_u *>(p + (size_t)k * kQuads);
  sums[slice][threadIdx.x & 15u] = sum;
  __syncthreads();
  if (slice != 0u) return;
#pragma unroll
  for (int k = 1; k < 16; ++k) sum += sums[k][threadIdx.x];
  const uint32_t ln = e & 63u, rest = e >> 6, tap = rest % 9u, ct = rest / 9u % CT, ot = rest / 9u / CT % OT, wt = rest / 9u / CT / OT;
  uint32_t cog, cig;
  P.div_cig.divmod(P.group0 + group, cog, cig);
  const uint32_t co = cog * (32u * OT) + ((wt & 1u) * OT + ot) * 16u + (ln >> 4) * 4u, ci = cig * (32u * CT) + ((wt >> 1) * CT + ct) * 16u + (ln & 15u);
  if (ci >= P.Cin) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (co + i >= P.Cout) break;
    float *d = P.dw + ((size_t)(co + i) * P.Cin + ci) * 9u + tap;
    *d = P.beta != 0.f ? *d + sum[i] : sum[i];
  }
}

static uint32_t ws_channel_tiles(uint32_t c) { return c <= 32u ? 1u : 2u; }

// The workgroups of a channel group: one per compute unit over all groups, no more than there are rows of octets.
static uint32_t ws_max_splits(uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W) {
  const uint32_t co = 32u * ws_channel_tiles(Cout), ci = 32u * ws_channel_tiles(Cin);
  const uint64_t groups = (uint64_t)((Cout + co - 1u) / co) * ((Cin + ci - 1u) / ci);
  const uint64_t most = (uint64_t)num_tiles * N * H * ((W + 7u) / 8u);
  return (uint32_t)std::max<uint64_t>(1u, std::min<uint64_t>(most, 256u / groups));
}

// a workgroup's sums
size_t conv3x3_wgrad_split_least_workspace(uint32_t Cin, uint32_t Cout) {
  return (size_t)ws_channel_tiles(Cout) * ws_channel_tiles(Cin) * 4u * 9u * 256u * 4u;
}
size_t conv3x3_wgrad_split_workspace(uint32_t num_tiles, uint32_t N, uint32_t Cin, uint32_t Cout, uint32_t H, uint32_t W) {
  const uint32_t ot = ws_channel_tiles(Cout), ct = ws_channel_tiles(Cin);
  const uint64_t groups = (uint64_t)((Cout + 32u * ot - 1u) / (32u * ot)) * ((Cin + 32u * ct - 1u) / (32u * ct));
  return (size_t)groups * ws_max_splits(num_tiles, N, Cin, Cout, H, W) * conv3x3_wgrad_split_least_workspace(Cin, Cout);
}

// at_once: channel groups whose sums the workspace holds
template <int OT, int CT>
static int launch_wgrad_split(WgradSplitParams P, uint32_t groups, uint32_t at_once, hipStream_t st) {
  for (P.group0 = 0u; P.group0 < groups; P.group0 += at_once) {
    const uint32_t n = std::min(at_once, groups - P.group0);
    hipLaunchKernelGGL((conv3x3_wgrad_split_kernel<OT, CT>), dim3(n * P.splits), dim3(kWsThreads), 0, st, P);
    hipLaunchKernelGGL((conv3x3_wgrad_split_reduce_kernel<OT, CT>), dim3(n * (4u * OT * CT * 9u * 64u / 16u)), dim3(256), 0, st, P);
    const int e = launch_status();
    if (e) return e;
  }
  return ADH_OK;
}

int conv3x3_wgrad_split(const Wgrad3x3Problem &q, void *workspace, size_t workspace_bytes, hipStream_t st) {
  WgradSplitParams P = {};
  for (uint32_t t = 0; t < q.num_tiles; ++t) {
    P.x[t] = reinterpret_cast<const float *>(q.x[t]);
    P.dy[t] = reinterpret_cast<const float *>(q.dy[t]);
  }
  P.part = reinterpret_cast<float *>(workspace);
  P.dw = q.dw;
  P.beta = q.beta;
  P.N = q.N; P.Cin = q.Cin; P.Cout = q.Cout; P.num_tiles = q.num_tiles;
  P.x_H = q.x_H; P.x_W = q.x_W; P.dy_H = q.dy_H; P.dy_W = q.dy_W;
  P.x_VH = q.x_H; P.dy_VH = q.dy_H;
  P.pad_r = q.pad_r; P.pad_c = q.pad_c;
  P.step = q.stacked ? q.dy_H : std::max(q.x_H, q.dy_H);
  P.neighbours = q.neighbours ? 1 : 0;
  if (q.stacked) {
    if ((uint64_t)q.dy_H * q.num_tiles >= (1ull << 31)) return ADH_EUNIMPL;
    P.x_VH = P.dy_VH = q.dy_H * q.num_tiles;
    P.last_tile = q.num_tiles - 1u;
  }
  const uint32_t NI = q.stacked ? q.N : q.N * q.num_tiles;
  const uint32_t OT = ws_channel_tiles(q.Cout), CT = ws_channel_tiles(q.Cin);
  // Column tiles of TW pixels by RS = 64 / TW rows a step: the fewest steps, a new run (an image's column tile: its first
  // rows are waited for) priced as three quarters of one, and narrower tiles for the columns they stage twice (a layer of
  // 64 channels on 56 x 56: seven tiles of 8 are 6 % fewer steps than two of 32 and take 0.077 ms against 0.059).
  double best = 1e300;
  for (uint32_t logQ = 3; logQ >= 1u; --logQ) {
    const uint32_t TW = 4u << logQ, RS = 64u / TW;
    const double cost = (double)NI * ((q.dy_W + TW - 1u) / TW) * ((P.dy_VH + RS - 1u) / RS + 0.75) * (logQ == 3u ? 1.0 : logQ == 2u ? 1.05 : 1.25);
    if (cost < best) {
      best = cost;
      P.logQ = logQ; P.TW = TW; P.RS = RS;
    }
  }
  P.NR = 2u * P.RS + 2u;
  P.x_row_bytes = (P.TW / 8u + 1u) * 32u * CT * 16u;
  P.dy_row_bytes = P.TW / 8u * 32u * OT * 16u;
  P.x_part_bytes = P.NR * P.x_row_bytes;
  P.dy_part_bytes = 2u * P.RS * P.dy_row_bytes;
  P.col_tiles = (q.dy_W + P.TW - 1u) / P.TW;
  P.row_steps = (P.dy_VH + P.RS - 1u) / P.RS;
  const uint64_t total = (uint64_t)NI * P.col_tiles * P.row_steps;
  if (total >= (1ull << 31)) return ADH_EUNIMPL;
  P.total_steps = (uint32_t)total;
  P.ci_groups = (q.Cin + 32u * CT - 1u) / (32u * CT);
  const uint32_t groups = P.ci_groups * ((q.Cout + 32u * OT - 1u) / (32u * OT));
  P.splits = std::min(ws_max_splits(q.num_tiles, q.N, q.Cin, q.Cout, q.dy_H, q.dy_W), P.total_steps);
  const uint64_t room = workspace_bytes / conv3x3_wgrad_split_least_workspace(q.Cin, q.Cout);  // for workgroups' sums
  if (room == 0u) return ADH_EWORKSPACE;
  const uint32_t at_once = (uint32_t)std::min<uint64_t>(groups, room);
  P.splits = (uint32_t)std::min<uint64_t>(P.splits, room / at_once);
  if ((uint64_t)groups * P.splits >= (1ull << 24)) return ADH_EUNIMPL;
  P.div_row_steps = FastDiv(P.row_steps); P.div_cols = FastDiv(P.col_tiles);
  P.div_N = FastDiv(q.N); P.div_step = FastDiv(P.step); P.div_splits = FastDiv(P.splits); P.div_cig = FastDiv(P.ci_groups);
  if (OT == 2u) return CT == 2u ? launch_wgrad_split<2, 2>(P, groups, at_once, st) : launch_wgrad_split<2, 1>(P, groups, at_once, st);
  return CT == 2u ? launch_wgrad_split<1, 2>(P, groups, at_once, st) : launch_wgrad_split<1, 1>(P, groups, at_once, st);
}

}  // namespace adh
