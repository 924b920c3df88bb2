// Filter gradient at stride 2 (3x3 with padding 1, or 1x1) over row tiles without halo, on the bf16 matrix cores, of fp32 tensors
// (three parts and six products, split_bf16.h) and of bf16 ones:
//   dw[co][ci][a][b] = beta*dw + sum over images, R, Q of dy[co][R][Q] * x[ci][2R + a - 1][2Q + b - 1]
//
// Mapping.  Per tap D[co][ci] += A[co][pixel] B[pixel][ci] on v_mfma_f32_16x16x32_bf16, k = 32 output pixels: four octets of
// neighbouring pixels of a row.
//   * A row of x lies in LDS as its even columns and its odd ones, [channel][pixel] each: the window's three columns are the odd
//     ones from the pixel before on (the octet and the dword before it, by v_alignbit), the even ones and the odd ones.
//   * A workgroup owns 16*OT*WO output channels x 16*WC input channels x all taps and a run of steps; a step is RS rows of TW
//     output columns, 32 pixels (1 x 32, 2 x 16 or 4 x 8).  A wave keeps 16*OT x 16 x taps sums.
//   * x rows go through a ring of 4 RS + 1 rows (2 RS new ones a step), dy rows through two buffers.  The rows of the next step are
//     stored while this one is multiplied, the ones after those are on their way in registers; of the two waves of a
//     SIMD one stages while the other multiplies.  One barrier a step.
//   * Past dy's last row dy is zero and x need not be there or finite: sums that come out as NaN are computed over again in plain
//     fp32 from the pixels that exist.
//   * The workgroups' sums are added by a second kernel in a fixed order (reproducible).
// Measured (32 images, 4 tiles; before: v_mfma_f32 kernels, in bf16 over widened values): fp32 3x3, 128 -> 256 channels on 16 x 64 tiles
// 0.202 -> 0.128 ms (150 TFLOP/s), 64 -> 128 on 32 x 128 0.217 -> 0.148, 256 -> 512 on 8 x 32 0.206 -> 0.129; bf16 3x3, 128 -> 256
// 0.341 -> 0.068, 1x1 0.143 -> 0.025; fp32 1x1, 128 -> 256 on 16 x 64 39 -> 33 us, 96 -> 96, 4 images, 8 tiles of 6 x 88, 19.5 -> 10.7, 24 shapes 0.68
// of the time (one workgroup per compute unit in place of two 50 and 10.8) at 0.2 - 0.5 of the error; 56 -> 112, 2 images, 2 tiles of 22 x 124: 36 -> 16 us.  Relative error against double
// precision over the former kernels': fp32 0.2 - 0.7 (up to 1.9 with the products below h*h in the same sums: six roundings a step in place of
// one, at no less time: 0.0 - 0.3 % of a projection block), bf16 0.35 - 1.0.
// Bound: fp32 by splitting and storing four rows' worth of x per output row beside 1728 matrix cycles a wave and step; bf16 by
// the staging alone; short layers by the workgroups' sums.
#include "conv_s2_wgrad.h"

#include <algorithm>
#include <cmath>

#include "wgrad_sums.h"

namespace adh {

struct S2WgParams : WgradSums {
  const void *x[ADH_MAX_TILES], *dy[ADH_MAX_TILES];
  uint32_t N;
  uint32_t dy_H, dy_W, x_H, x_W, dy_VH, last_tile;
  uint32_t logT, TW, RS, NR, swizzle;  // TW = 1 << logT; swizzle: dy's octets of channel c are exchanged by c >> swizzle
  uint32_t row_steps, total_steps, ci_groups;
  FastDiv div_row_steps, div_cols, div_H, div_splits;
};

constexpr uint32_t s2wg_ring(uint32_t rs, int taps) { return taps == 9 ? 4u * rs + 1u : 2u * rs; }
// elements of a channel's row: the even columns, room for the odd one before the first, the odd columns
constexpr uint32_t s2wg_pitch(uint32_t tw, int taps) { return taps == 9 ? 2u * tw + 8u : tw + 8u; }
// the narrowest step: three parts of 4 x 8 ones do not fit the LDS (64 channels), or only once (32)
constexpr uint32_t s2wg_narrowest(int taps, int parts) { return taps == 9 && parts == 3 ? 16u : 8u; }
// of one part, over the shapes of a step
constexpr uint32_t s2wg_x_bytes(int taps, uint32_t ci, int parts) {
  uint32_t most = 0;
  for (uint32_t tw = s2wg_narrowest(taps, parts); tw <= 32u; tw *= 2u) {
    const uint32_t b = s2wg_ring(32u / tw, taps) * ci * s2wg_pitch(tw, taps) * 2u;
    most = b > most ? b : most;
  }
  return most;
}

// eight neighbouring columns of x and four of dy, as loaded
template <typename T> struct S2Raw;
template <> struct S2Raw<float> { floatx4 x[2], dy; };
template <> struct S2Raw<uint16_t> { uintx4 x; uintx2 dy; };
typedef uintx4 s2_u32x4 __attribute__((aligned(2)));
typedef uintx2 s2_u32x2 __attribute__((aligned(2)));

template <typename T, int TAPS, int OT, int WO, int WC>
__global__ __launch_bounds__(64 * WO * WC, 2) void conv_s2_wgrad_kernel(const S2WgParams P) {
  constexpr uint32_t THREADS = 64u * WO * WC, CO = 16u * OT * WO, CI = 16u * WC;
  constexpr int PARTS = sizeof(T) == 4 ? 3 : 1;
  constexpr uint32_t XB = s2wg_x_bytes(TAPS, CI, PARTS), DB = 2u * CO * 32u * 2u;  // bytes of one part
  constexpr uint32_t ROWS = TAPS == 9 ? 2u : 1u;                            // new x rows per output row
  constexpr int XU = (int)((ROWS * CI * 8u + THREADS - 1u) / THREADS);      // units of eight columns a thread stages per step
  constexpr int DU = (int)((CO * 8u + THREADS - 1u) / THREADS);             // and of four of dy
  __shared__ __align__(16) char lds[PARTS * (XB + DB)];
  __shared__ uint32_t nan_sums;
  char *const dyl = lds + PARTS * XB;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t wo = wave % WO, wc = wave / WO;

  uint32_t group, split, cog, cig;
  P.div_splits.divmod(blockIdx.x, group, split);
  P.div_cig.divmod(group, cog, cig);
  const uint32_t co0 = cog * CO, ci0 = cig * CI;
  uint32_t s = (uint32_t)((uint64_t)P.total_steps * split / P.splits);
  const uint32_t s_end = (uint32_t)((uint64_t)P.total_steps * (split + 1u) / P.splits);
  if (tid == 0u) nan_sums = 0u;

  const uint32_t TW = P.TW, pitch = s2wg_pitch(TW, TAPS);
  const size_t x_plane = (size_t)P.x_H * P.x_W, dy_plane = (size_t)P.dy_H * P.dy_W;
  uint32_t n = 0, c0 = 0;  // the run that the workgroup stands in: an image and a column tile of it
  const int32_t xW = (int32_t)P.x_W, dW = (int32_t)P.dy_W;

  // Staging: units of eight x columns and of four dy columns, columns first, then channels, then rows (a wave's units are of one row).
  const uint32_t log_u = P.logT - 2u, xq = tid & ((1u << log_u) - 1u);  // units of a row: TW / 4 for either
  const uint32_t x_c = (tid >> log_u) & (CI - 1u), dy_c = (tid >> log_u) & (CO - 1u);
  const uint32_t x_row = (wave * 64u) >> log_u >> __builtin_ctz(CI), dy_row = (wave * 64u) >> log_u >> __builtin_ctz(CO);
  const uint32_t x_rows = THREADS >> log_u >> __builtin_ctz(CI), dy_rows = THREADS >> log_u >> __builtin_ctz(CO);  // per unit of a thread
  const bool x_ok = ci0 + x_c < P.Cin, dy_ok = co0 + dy_c < P.Cout;
  const uint32_t tail_c = tid & (CI - 1u), tail_row = tid >> __builtin_ctz(CI);
  const bool tail_ok = ci0 + tail_c < P.Cin;
  const size_t x_chan = (size_t)(x_ok ? ci0 + x_c : 0u) * x_plane, dy_chan = (size_t)(dy_ok ? co0 + dy_c : 0u) * dy_plane;
  const size_t tail_chan = (size_t)(tail_ok ? ci0 + tail_c : 0u) * x_plane;
  S2Raw<T> raw[XU > DU ? XU : DU];
  T tail = 0;

  auto x_at = [&](uint32_t r) {  // row r of the stacked tensor
    const uint32_t t = min(P.div_H.div(r >> 1), P.last_tile);
    return (const ADH_GLOBAL T *)P.x[t] + ((size_t)n * P.Cin * x_plane + (size_t)(r - t * P.x_H) * P.x_W);
  };
  auto dy_at = [&](uint32_t R) {
    const uint32_t t = min(P.div_H.div(R), P.last_tile);
    return (const ADH_GLOBAL T *)P.dy[t] + ((size_t)n * P.Cout * dy_plane + (size_t)(R - t * P.dy_H) * P.dy_W);
  };
  // Values from column Q of a row of W on, loaded from where all exist; what lies past the row's end is zero.
  auto load_x8 = [&](const ADH_GLOBAL T *row, int32_t Q, S2Raw<T> &v) {
    if constexpr (PARTS == 3) {
      v.x[0] = *(const ADH_GLOBAL floatx4_u *)(row + min(Q, xW - 4));
      v.x[1] = *(const ADH_GLOBAL floatx4_u *)(row + min(Q + 4, xW - 4));
    } else {
      v.x = *(const ADH_GLOBAL s2_u32x4 *)(row + min(Q, xW - 8));
    }
  };
  auto load_dy4 = [&](const ADH_GLOBAL T *row, int32_t Q, S2Raw<T> &v) {
    if constexpr (PARTS == 3) v.dy = *(const ADH_GLOBAL floatx4_u *)(row + min(Q, dW - 4));
    else v.dy = *(const ADH_GLOBAL s2_u32x2 *)(row + min(Q, dW - 4));
  };
  const int32_t x_vh = (int32_t)(2u * P.dy_VH);
  // x rows x0 .. x0 + nx - 1 (row i of a 1x1 window: x0 + 2 i), dy rows d0 .. d0 + nd - 1
  auto load = [&](int32_t x0, uint32_t nx, uint32_t d0, uint32_t nd) {
    const int32_t Qx = (int32_t)(2u * c0 + 8u * xq), Qd = (int32_t)(c0 + 4u * xq);
#pragma unroll
    for (int j = 0; j < XU; ++j) {
      const uint32_t i = (uint32_t)j * x_rows + x_row;
      const int32_t r = x0 + (int32_t)(TAPS == 9 ? i : 2u * i);
      if (i < nx) load_x8(x_at((uint32_t)min(max(r, 0), x_vh - 1)) + x_chan, Qx, raw[j]);
    }
#pragma unroll
    for (int j = 0; j < DU; ++j) {
      const uint32_t i = (uint32_t)j * dy_rows + dy_row;
      if (i < nd) load_dy4(dy_at(min(d0 + i, P.dy_VH - 1u)) + dy_chan, Qd, raw[j]);
    }
    if (TAPS == 9 && tail_row < nx) {
      const int32_t r = x0 + (int32_t)tail_row;
      tail = (x_at((uint32_t)min(max(r, 0), x_vh - 1)) + tail_chan)[c0 ? 2u * c0 - 1u : 0u];
    }
  };
  // slot0: ring slot of x row x0; buf: the dy buffer
  auto store = [&](int32_t x0, uint32_t nx, uint32_t slot0, uint32_t d0, uint32_t nd, uint32_t buf) {
    auto slot_of = [&](uint32_t i) {
      const uint32_t slot = slot0 + i;
      return slot - (slot >= P.NR ? P.NR : 0u);
    };
    const int32_t Qx = (int32_t)(2u * c0 + 8u * xq), Qd = (int32_t)(c0 + 4u * xq);
#pragma unroll
    for (int j = 0; j < XU; ++j) {
      const uint32_t i = (uint32_t)j * x_rows + x_row;
      if (i < nx) {
        const int32_t r = x0 + (int32_t)(TAPS == 9 ? i : 2u * i);
        const bool ok = x_ok && r >= 0 && r < x_vh;
        char *p = lds + (slot_of(i) * CI + x_c) * (pitch * 2u) + 8u * xq;
        if constexpr (PARTS == 3) {
          floatx4 even, odd;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int32_t q = Qx + 4 * h, d = q - min(q, xW - 4);  // (even; 4 and more: none exists)
            floatx4 v = raw[j].x[h];
            if (d == 2) v = floatx4{v[2], v[3], 0.f, 0.f};
            if (!ok || d >= 4) v = floatx4{0.f, 0.f, 0.f, 0.f};
            even[2 * h] = v[0]; even[2 * h + 1] = v[2];
            odd[2 * h] = v[1]; odd[2 * h + 1] = v[3];
          }
          uint32_t part[3][2];
          split_pair(even[0], even[1], part[0][0], part[1][0], part[2][0]);
          split_pair(even[2], even[3], part[0][1], part[1][1], part[2][1]);
#pragma unroll
          for (int k = 0; k < 3; ++k) *reinterpret_cast<uintx2 *>(p + k * XB) = uintx2{part[k][0], part[k][1]};
          if constexpr (TAPS == 9) {
            split_pair(odd[0], odd[1], part[0][0], part[1][0], part[2][0]);
            split_pair(odd[2], odd[3], part[0][1], part[1][1], part[2][1]);
#pragma unroll
            for (int k = 0; k < 3; ++k) *reinterpret_cast<uintx2 *>(p + k * XB + (TW + 8u) * 2u) = uintx2{part[k][0], part[k][1]};
          }
        } else {
          const int32_t d = Qx - min(Qx, xW - 8);
          uintx4 v = raw[j].x;
          if (d >= 4) v = uintx4{v[2], v[3], 0u, 0u};
          if (d & 2) v = uintx4{v[1], v[2], v[3], 0u};
          if (!ok || d >= 8) v = uintx4{0u, 0u, 0u, 0u};
          *reinterpret_cast<uintx2 *>(p) = uintx2{__builtin_amdgcn_perm(v[1], v[0], 0x05040100u), __builtin_amdgcn_perm(v[3], v[2], 0x05040100u)};
          if constexpr (TAPS == 9)
            *reinterpret_cast<uintx2 *>(p + (TW + 8u) * 2u) = uintx2{__builtin_amdgcn_perm(v[1], v[0], 0x07060302u), __builtin_amdgcn_perm(v[3], v[2], 0x07060302u)};
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < DU; ++j) {
      const uint32_t i = (uint32_t)j * dy_rows + dy_row;
      if (i < nd) {
        const int32_t d = Qd - min(Qd, dW - 4);
        const bool none = !dy_ok || d0 + i >= P.dy_VH || d >= 4;
        const uint32_t oct = (xq >> 1) ^ ((dy_c >> P.swizzle) & ((TW >> 3) - 1u));
        char *p = dyl + (((buf * P.RS + i) * CO + dy_c) * TW + oct * 8u + (xq & 1u) * 4u) * 2u;
        if constexpr (PARTS == 3) {
          floatx4 v = raw[j].dy;
#pragma unroll
          for (int k = 1; k < 4; ++k) v = floatx4{d >= k ? v[1] : v[0], d >= k ? v[2] : v[1], d >= k ? v[3] : v[2], d >= k ? 0.f : v[3]};
          if (none) v = floatx4{0.f, 0.f, 0.f, 0.f};
          uint32_t part[3][2];
          split_pair(v[0], v[1], part[0][0], part[1][0], part[2][0]);
          split_pair(v[2], v[3], part[0][1], part[1][1], part[2][1]);
#pragma unroll
          for (int k = 0; k < 3; ++k) *reinterpret_cast<uintx2 *>(p + k * DB) = uintx2{part[k][0], part[k][1]};
        } else {
          const uint64_t v = none ? 0u : ((uint64_t)raw[j].dy[1] << 32 | raw[j].dy[0]) >> (16 * d);
          *reinterpret_cast<uintx2 *>(p) = uintx2{(uint32_t)v, (uint32_t)(v >> 32)};
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (TAPS == 9 && tail_row < nx) {
      const int32_t r = x0 + (int32_t)tail_row;
      const bool ok = tail_ok && c0 > 0u && r >= 0 && r < x_vh;
      uint16_t *p = reinterpret_cast<uint16_t *>(lds + (slot_of(tail_row) * CI + tail_c) * (pitch * 2u) + (TW + 7u) * 2u);
      if constexpr (PARTS == 3) {
        uint32_t h, m, l;
        split_pair(ok ? tail : 0.f, 0.f, h, m, l);
        p[0] = (uint16_t)h;
        p[XB / 2u] = (uint16_t)m;
        p[XB] = (uint16_t)l;
      } else {
        p[0] = ok ? tail : (uint16_t)0;
      }
    }
  };

  // ---- this lane group's octet of a step: row io of the step, octet qo of the row ----
  const uint32_t io = g >> (P.logT - 3u), qo = g & ((TW >> 3) - 1u);
  const uint32_t a_c = wo * OT * 16u + l16;
  const uint32_t b_base = ((wc * 16u + l16) * pitch + 8u * qo) * 2u;

  floatx4 acc[OT][TAPS], low[PARTS == 3 ? OT : 1][PARTS == 3 ? TAPS : 1];  // (fp32: low, the products below h*h)
#pragma unroll
  for (int ot = 0; ot < OT; ++ot)
#pragma unroll
    for (int t = 0; t < TAPS; ++t) {
      acc[ot][t] = floatx4{0.f, 0.f, 0.f, 0.f};
      if constexpr (PARTS == 3) low[ot][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

  // base: ring slot of the step's first x row
  auto multiply = [&](uint32_t base, uint32_t buf) {
    uintx4 a[OT][PARTS];
#pragma unroll
    for (int ot = 0; ot < OT; ++ot) {
      const uint32_t c = a_c + ot * 16u, oct = qo ^ ((c >> P.swizzle) & ((TW >> 3) - 1u));
#pragma unroll
      for (int k = 0; k < PARTS; ++k)
        a[ot][k] = *reinterpret_cast<const uintx4 *>(dyl + k * DB + (((buf * P.RS + io) * CO + c) * TW + oct * 8u) * 2u);
    }
#pragma unroll
    for (int r = 0; r < (TAPS == 9 ? 3 : 1); ++r) {
      uint32_t slot = base + (TAPS == 9 ? 2u * io + (uint32_t)r : io);
      slot -= slot >= P.NR ? P.NR : 0u;
      const char *p = lds + slot * (CI * 2u) * pitch + b_base;
      constexpr int COLS = TAPS == 9 ? 3 : 1;
      uintx4 w[PARTS][COLS];
#pragma unroll
      for (int k = 0; k < PARTS; ++k) {
        const uintx4 even = *reinterpret_cast<const uintx4 *>(p + k * XB);
        if constexpr (TAPS == 9) {
          const uintx4 d = *reinterpret_cast<const uintx4 *>(p + k * XB + (TW + 8u) * 2u);
          const uint32_t e = *reinterpret_cast<const uint32_t *>(p + k * XB + (TW + 6u) * 2u);
          w[k][0] = uintx4{__builtin_amdgcn_alignbit(d[0], e, 16), __builtin_amdgcn_alignbit(d[1], d[0], 16),
                           __builtin_amdgcn_alignbit(d[2], d[1], 16), __builtin_amdgcn_alignbit(d[3], d[2], 16)};
          w[k][1] = even;
          w[k][2] = d;
        } else {
          w[k][0] = even;
        }
      }
      auto products = [&](auto &sum, int ka, int kb) {
#pragma unroll
        for (int col = 0; col < COLS; ++col)
#pragma unroll
          for (int ot = 0; ot < OT; ++ot) sum[ot][r * 3 + col] = mfma_bf16(a[ot][ka], w[kb][col], sum[ot][r * 3 + col]);
      };
      if constexpr (PARTS == 3) {
        products(low, 0, 2); products(low, 1, 1); products(low, 2, 0); products(low, 0, 1); products(low, 1, 0);
      }
      products(acc, 0, 0);
    }
  };

  while (s < s_end) {
    // a run: steps of one image and column tile
    uint32_t run, rs, ctile;
    P.div_row_steps.divmod(s, run, rs);
    P.div_cols.divmod(run, n, ctile);
    c0 = ctile * TW;
    const uint32_t steps = min(s_end - s, P.row_steps - rs);
    uint32_t R = rs * P.RS, base = 0, buf = 0;
    const uint32_t lead = TAPS == 9 ? 1u : 0u, nx = ROWS * P.RS;  // rows before a step's new ones
    int32_t x0 = (int32_t)(2u * R) - (int32_t)lead;               // the step's first x row
    if (lead) load(x0, 1u, 0u, 0u);
    lds_barrier();  // every wave is done with the run before
    if (lead) store(x0, 1u, 0u, 0u, 0u, 0u);
    load(x0 + (int32_t)lead, nx, R, P.RS);
    store(x0 + (int32_t)lead, nx, lead, R, P.RS, 0u);
    if (steps > 1u) load(x0 + (int32_t)(lead + 2u * P.RS), nx, R + P.RS, P.RS);
    lds_barrier();
    for (uint32_t k = 0; k < steps; ++k) {
      auto stage = [&]() {
        if (k + 1u < steps) {
          uint32_t slot = base + nx + lead;
          slot -= slot >= P.NR ? P.NR : 0u;
          store(x0 + (int32_t)(lead + 2u * P.RS), nx, slot, R + P.RS, P.RS, buf ^ 1u);
          if (k + 2u < steps) load(x0 + (int32_t)(lead + 4u * P.RS), nx, R + 2u * P.RS, P.RS);
        }
      };
      const bool first = wave < WO * WC / 2;
      if (first) stage();
      __builtin_amdgcn_sched_barrier(0);
      multiply(base, buf);
      __builtin_amdgcn_sched_barrier(0);
      if (!first) stage();
      R += P.RS;
      x0 += (int32_t)(2u * P.RS);
      base += nx;
      base -= base >= P.NR ? P.NR : 0u;
      buf ^= 1u;
      if (k + 1u < steps) lds_barrier();
    }
    s += steps;
  }

  // ---- the sums to the workspace ----
  constexpr uint32_t kWave = OT * TAPS * 256u;
  float *const part = P.part + (size_t)blockIdx.x * (WO * WC * kWave);
  ADH_GLOBAL float *out = (ADH_GLOBAL float *)part + (size_t)wave * kWave + lane * 4u;
  bool nan = false;
#pragma unroll
  for (int ot = 0; ot < OT; ++ot)
#pragma unroll
    for (int t = 0; t < TAPS; ++t) {
      floatx4 sum = acc[ot][t];
      if constexpr (PARTS == 3) sum += low[ot][t];
      nan |= __builtin_isunordered(sum[0], sum[1]) || __builtin_isunordered(sum[2], sum[3]);
      *(ADH_GLOBAL floatx4_u *)(out + (ot * TAPS + t) * 256) = sum;
    }
  if (nan) nan_sums = 1u;
  __syncthreads();
  if (nan_sums == 0u) return;
  // sums that are NaN once more in plain fp32, straight from memory
  auto value = [](T v) {
    if constexpr (PARTS == 3) return v;
    else return bf16_bits_to_f32(v);
  };
  s = (uint32_t)((uint64_t)P.total_steps * split / P.splits);
  for (uint32_t at = tid; at < WO * WC * kWave; at += THREADS) {
    if (part[at] == part[at]) continue;
    const uint32_t i = at & 3u, ln = at >> 2 & 63u, rest = at >> 8, tap = rest % TAPS, ot = rest / TAPS % OT, wt = rest / TAPS / OT;
    const uint32_t co = co0 + ((wt % WO) * OT + ot) * 16u + (ln >> 4) * 4u + i, ci = ci0 + (wt / WO) * 16u + (ln & 15u);
    float sum = 0.f;
    if (co < P.Cout && ci < P.Cin)
      for (uint32_t st = s; st < s_end && sum == sum; ++st) {  // (a NaN stays one)
        uint32_t run, rs, ctile;
        P.div_row_steps.divmod(st, run, rs);
        P.div_cols.divmod(run, n, ctile);
        for (uint32_t R = rs * P.RS; R < min((rs + 1u) * P.RS, P.dy_VH) && sum == sum; ++R)
          for (uint32_t Q = ctile * TW; Q < min((ctile + 1u) * TW, P.dy_W) && sum == sum; ++Q) {
            const int32_t xr = (int32_t)(2u * R) + (TAPS == 9 ? (int32_t)(tap / 3u) - 1 : 0), xc = (int32_t)(2u * Q) + (TAPS == 9 ? (int32_t)(tap % 3u) - 1 : 0);
            float xe = 0.f;
            if (xr >= 0 && xr < x_vh && xc >= 0 && xc < xW) xe = value((x_at((uint32_t)xr) + (size_t)ci * x_plane)[xc]);
            sum = __builtin_fmaf(value((dy_at(R) + (size_t)co * dy_plane)[Q]), xe, sum);
          }
      }
    part[at] = sum;
  }
}

// ---- host side ----

struct S2WgPlan {
  S2WgParams P;
  bool co64, ci64;
  uint32_t groups;
  size_t split_bytes;  // a split's sums over all channel groups
};

static bool s2wg_plan(const S2WgradProblem &q, S2WgPlan *plan) {
  S2WgParams &P = plan->P;
  if (q.dy_W < 4u || (uint64_t)q.dy_H * q.num_tiles * 2u >= (1ull << 31)) return false;
  if ((uint64_t)q.Cin * q.Cout * 9u >= (1ull << 31)) return false;
  P.N = q.N; P.Cin = q.Cin; P.Cout = q.Cout;
  P.dy_H = q.dy_H; P.dy_W = q.dy_W; P.x_H = 2u * q.dy_H; P.x_W = 2u * q.dy_W;
  P.dy_VH = q.dy_H * q.num_tiles;
  P.last_tile = q.num_tiles - 1u;
  P.beta = q.beta;
  // the step's shape: the fewest steps, a new run (its first rows are waited for) priced as one, narrower ones for the rows and
  // columns that they stage twice
  double best = 1e300;
  plan->co64 = q.Cout > 32u; plan->ci64 = q.Cin > 32u;
  const uint32_t co = plan->co64 ? 64u : 32u, ci = plan->ci64 ? 64u : 32u;
  for (uint32_t logT = 5; 1u << logT >= s2wg_narrowest(q.taps, q.dtype == ADH_F32 ? 3 : 1); --logT) {
    const uint32_t TW = 1u << logT, RS = 32u / TW;
    const double cost = (double)q.N * ((q.dy_W + TW - 1u) / TW) * ((P.dy_VH + RS - 1u) / RS + 1.0) * (logT == 5u ? 1.0 : logT == 4u ? 1.03 : 1.1);
    if (cost >= best) continue;
    best = cost;
    P.logT = logT; P.TW = TW; P.RS = RS;
  }
  P.NR = s2wg_ring(P.RS, q.taps);
  P.swizzle = 7u - P.logT;  // channels whose rows of dy fill 256 bytes
  P.row_steps = (P.dy_VH + P.RS - 1u) / P.RS;
  const uint32_t cols = (q.dy_W + P.TW - 1u) / P.TW;
  const uint64_t total = (uint64_t)q.N * cols * P.row_steps;
  if (total >= (1ull << 31)) return false;
  P.total_steps = (uint32_t)total;
  P.ci_groups = (q.Cin + ci - 1u) / ci;
  plan->groups = P.ci_groups * ((q.Cout + co - 1u) / co);
  plan->split_bytes = (size_t)plan->groups * co * ci * q.taps * 4u;
  // One workgroup per compute unit over all groups (two where the registers and the LDS hold them: a projection block of 80 -> 80 channels
  // on 4 tiles of 56 x 102 in bf16 takes 153 us with one of 64 x 64 channels and 169 with two, which run in turn), and no more than the reduction kernel pays for: the
  // square root is where a step's time saved is a split's sums added (8 to 60 in place of 25: 0 to 6 % slower).
  const bool both = plan->co64 && plan->ci64, twice = q.taps == 1 || (q.dtype == ADH_BF16 ? !both : !plan->co64 && !plan->ci64);
  const uint32_t most = twice ? 512u : 256u;
  P.splits = std::min(most / std::min(plan->groups, most), std::min(P.total_steps, (uint32_t)std::sqrt(25.0 * P.total_steps)));
  if ((uint64_t)plan->groups * P.splits >= (1ull << 22)) return false;
  P.div_row_steps = FastDiv(P.row_steps); P.div_cols = FastDiv(cols); P.div_H = FastDiv(P.dy_H); P.div_cig = FastDiv(P.ci_groups);
  return true;
}

size_t conv_s2_wgrad_workspace(const S2WgradProblem &q) {
  S2WgPlan plan = {};
  return s2wg_plan(q, &plan) ? (plan.split_bytes * plan.P.splits + 255u) & ~(size_t)255u : 0u;
}

size_t conv_s2_wgrad_required(const S2WgradProblem &q) {
  if (q.dtype != ADH_F32 || q.taps != 9 || q.N == 0 || q.dy_H == 0 || q.dy_W == 0) return 0;
  if (q.dy_W != 8u && q.dy_W % 16u != 0u) return 0;
  const uint32_t cols = std::min(q.dy_W, 16u);
  uint32_t rows = std::min(q.dy_H, 32u / cols);
  while (rows > 1u && q.dy_H % rows != 0u) --rows;
  if ((32u / cols) % rows != 0u) return 0;
  const uint32_t images = 32u / (cols * rows);
  if (images * (2u * rows + 1u) * (2u * cols + 1u) > 192u) return 0;
  if ((uint64_t)q.Cin * q.Cout * 9u >= (1ull << 31) || (uint64_t)q.N * q.Cin * q.dy_H * q.dy_W * 4u >= (1ull << 31)) return 0;
  const uint64_t chunks = (uint64_t)q.num_tiles * ((q.N + images - 1u) / images) * (q.dy_H / rows) * (q.dy_W / cols);
  if (chunks >= (1ull << 31)) return 0;
  const uint32_t groups = ((q.Cout + 63u) / 64u) * ((q.Cin + 31u) / 32u);
  const uint32_t most = std::max(1u, std::min((uint32_t)chunks / 4u, (512u + groups - 1u) / groups));
  const uint32_t per_split = ((uint32_t)chunks + most - 1u) / most;
  return (size_t)(((uint32_t)chunks + per_split - 1u) / per_split) * 9u * q.Cout * q.Cin * sizeof(float);
}

template <typename T, int TAPS, int OT, int WO, int WC>
static void launch_s2wg(const S2WgPlan &plan, hipStream_t st) {
  hipLaunchKernelGGL((conv_s2_wgrad_kernel<T, TAPS, OT, WO, WC>), dim3(plan.groups * plan.P.splits), dim3(64 * WO * WC), 0, st, plan.P);
  hipLaunchKernelGGL((wgrad_sums_kernel<TAPS, OT, WO, WC>), dim3(plan.groups * (WO * WC * OT * TAPS * 64u / 16u)), dim3(256), 0, st, static_cast<const WgradSums &>(plan.P));
}
template <typename T, int TAPS>
static void launch_s2wg_channels(const S2WgPlan &plan, hipStream_t st) {
  if (plan.co64) plan.ci64 ? launch_s2wg<T, TAPS, 2, 2, 4>(plan, st) : launch_s2wg<T, TAPS, 1, 4, 2>(plan, st);
  else plan.ci64 ? launch_s2wg<T, TAPS, 1, 2, 4>(plan, st) : launch_s2wg<T, TAPS, 1, 2, 2>(plan, st);
}

int conv_s2_wgrad(const S2WgradProblem &q, void *workspace, size_t workspace_bytes, hipStream_t st) {
  S2WgPlan plan = {};
  if (!s2wg_plan(q, &plan) || workspace_bytes < plan.split_bytes) return ADH_EUNIMPL;
  S2WgParams &P = plan.P;
  P.splits = (uint32_t)std::min<uint64_t>(P.splits, workspace_bytes / plan.split_bytes);
  P.div_splits = FastDiv(P.splits);
  for (uint32_t t = 0; t < q.num_tiles; ++t) {
    P.x[t] = q.x[t];
    P.dy[t] = q.dy[t];
  }
  P.part = reinterpret_cast<float *>(workspace);
  P.dw = q.dw;
  if (q.dtype == ADH_F32) q.taps == 9 ? launch_s2wg_channels<float, 9>(plan, st) : launch_s2wg_channels<float, 1>(plan, st);
  else q.taps == 9 ? launch_s2wg_channels<uint16_t, 9>(plan, st) : launch_s2wg_channels<uint16_t, 1>(plan, st);
  return launch_status();
}

}  // namespace adh
