// Filter gradient of the 3x3 stride-1 window over bf16 tensors on the matrix cores, over padded tiles or row tiles without halo, at any
// width from eight and any number of channels:
//   dw[co][ci][a][b] = beta*dw + sum over images, R, Q of dy[co][R][Q] * x[ci][R + a - halo][Q + b - halo]
//
// Mapping.  Per tap D[co][ci] += A[co][pixel] B[pixel][ci] on v_mfma_f32_16x16x32_bf16, k = 32 pixels: four octets of neighbouring
// pixels of a row.
//   * A workgroup owns 16*OT*WO output channels x 16*WC input channels x all taps and a run of steps; a step is RS rows of TW output
//     columns, 64 pixels (1 x 64 .. 8 x 8).  A wave keeps 16*OT x 16 x 9 sums: the octets of x that it shifts for
//     the three columns of a window's row feed 3*OT products.  Unlike a walk down whole columns of an image this splits small and narrow
//     images over the chip as finely as their sums are worth, and has no columns beyond an image's end to speak of.
//   * x rows go through a ring: a row is read once per run (an image's column of steps), its two columns behind the step's twice.  Rows
//     are loaded from wherever they start (2 bytes' alignment), so that neither odd widths nor missing halos want copies.
//   * Rows lie in LDS as [octet][channel], exchanged so that neither side's accesses meet in a bank (with channels 144 bytes apart
//     half of all cycles went there).  A step's rows are asked for two steps ahead, stored one ahead.  One barrier a step.
//   * Past dy's last row and column dy is zero and x need not be there or finite: sums that come out as NaN are computed over again in
//     plain fp32 from the pixels that exist.
//   * The workgroups' sums are added by a second kernel in a fixed order (reproducible).
// Measured, both kernels and, at odd widths before, the copies (before: conv3x3_bf16_wgrad.hip alone), us: 512 -> 512 channels, 32 images,
// 4 tiles of 4 x 16 575 -> 147; 128 -> 128, 8 images, 4 tiles of 64 x 255 243 -> 165 (920 TFLOP/s); 208 -> 433, 27 images, 3 tiles of
// 9 x 16 218 -> 110; 18 -> 16, 2 tiles of 42 x 24 40 -> 9; 900 layers of 16 to 512 channels 1.62 times as fast (geometric mean).
// Relative error against double precision over the former kernel's in those: 0.61 in the mean, nowhere above 1 (steps_plan).
// Bound: long layers by the waits between a step's LDS accesses, products and staging (two workgroups a compute unit, 40 % of the
// matrix cores' cycles); short ones by the two launches and the sums.
#include "conv3x3_wgrad_steps.h"

#include <algorithm>
#include <cmath>

#include "wgrad_sums.h"

namespace adh {

struct StepsParams : WgradSums {
  const void *x[ADH_MAX_TILES], *dy[ADH_MAX_TILES];
  uint32_t N, stacked, by_xcd;
  uint32_t H, W, x_H, x_W;         // a tile's dy and x
  uint32_t rows, x_rows;           // of a plane (an image; stacked: of all tiles): of dy and x
  uint32_t row_steps, cols, total_steps, ci_groups;
  uint32_t chain;  // (HI) steps whose products go into one chain of additions
  FastDiv div_row_steps, div_cols, div_H, div_N, div_groups, div_splits;
};

constexpr uint32_t kStepBlocks = 2;  // k blocks (of 32 pixels) a step
// the ring holds a step's rows and the most that the next one brings (its run may be another)
constexpr uint32_t steps_ring(uint32_t rs) { return 2u * rs + 4u; }
// the narrowest step of 32 channels: a wave's units of eight columns are of one row
constexpr uint32_t steps_narrowest(bool few) { return few ? 16u : 8u; }
// x rows with an octet behind them (whose first two columns exist), dy rows, twice
constexpr uint32_t steps_x_bytes(uint32_t tw, uint32_t ci) { return steps_ring(kStepBlocks * 32u / tw) * (tw / 8u + 1u) * ci * 16u; }
constexpr uint32_t steps_dy_bytes(uint32_t co) { return 2u * kStepBlocks * 4u * co * 16u; }
// How THREADS threads take a row's units of eight columns, columns first, then channels, then rows (a wave's units are of one row):
// unit j of a thread is channel pass j % passes of row (j / passes) * rows + the thread's.
template <uint32_t THREADS, uint32_t U, uint32_t C>
struct StepsUnits {
  static constexpr uint32_t passes = U * C > THREADS ? U * C / THREADS : 1u, channels = C / passes, rows = THREADS / (U * channels);
  static constexpr int count(uint32_t n) { return (int)((n + rows - 1u) / rows * passes); }  // units that cover n rows
  static constexpr int sure(uint32_t n) { return (int)(n / rows * passes); }                 // units that every thread has of n rows
  uint32_t c, row, q;
  __device__ StepsUnits(uint32_t tid, uint32_t wave) : c(tid / U % channels), row(wave * 64u / (U * channels)), q(tid % U) {}
  __device__ uint32_t channel(int j) const { return (uint32_t)j % passes * channels + c; }
  __device__ uint32_t row_of(int j) const { return (uint32_t)j / passes * rows + row; }
};

typedef uintx4 steps_u32x4 __attribute__((aligned(2)));
typedef uint32_t steps_u32 __attribute__((aligned(2)));

// Values from column Q on of a row of W were loaded from column min(max(Q, 0), W - 8) on: to their places, zeros
// where none exists.
__device__ __forceinline__ uintx4 steps_place(uintx4 v, int32_t Q, int32_t W) {
  const int32_t d = Q - min(max(Q, 0), W - 8);
  if (d != 0) {
    if (d < 0) {
      v = uintx4{v[0] << 16, __builtin_amdgcn_alignbit(v[1], v[0], 16), __builtin_amdgcn_alignbit(v[2], v[1], 16), __builtin_amdgcn_alignbit(v[3], v[2], 16)};
    } else {
      if (d & 4) v = uintx4{v[2], v[3], 0u, 0u};
      if (d & 2) v = uintx4{v[1], v[2], v[3], 0u};
      if (d & 1) v = uintx4{__builtin_amdgcn_alignbit(v[1], v[0], 16), __builtin_amdgcn_alignbit(v[2], v[1], 16), __builtin_amdgcn_alignbit(v[3], v[2], 16), v[3] >> 16};
      if (d >= 8) v = uintx4{0u, 0u, 0u, 0u};
    }
  }
  return v;
}

// A step: RS rows of TW columns.  HI: a chain's sums are added to others, and what that addition rounds off begins the next chain, so that
// hi + acc is the exact sum of the chains, and a split may be of any number of them (16 output channels a wave: 72 sums and as many
// others are more registers than there are).
template <uint32_t TW, int OT, int WO, int WC, bool HI>
__global__ __launch_bounds__(64 * WO * WC, HI ? 2 : OT == 4 || (OT == 2 && WC == 4 && TW == 64u) ? 2 : OT == 2 ? 3 : 4) void conv3x3_wgrad_steps_kernel(const StepsParams P) {
  constexpr uint32_t THREADS = 64u * WO * WC, CO = 16u * OT * WO, CI = 16u * WC;
  constexpr uint32_t KB = kStepBlocks, RS = KB * 32u / TW, NR = steps_ring(RS), U = TW / 8u;
  constexpr uint32_t XB = steps_x_bytes(TW, CI);
  typedef StepsUnits<THREADS, U, CI> XUnits;
  typedef StepsUnits<THREADS, U, CO> DyUnits;
  // units that a thread stages per step (x: of all rows, where a run begins), and the two columns behind
  constexpr int XU = XUnits::count(RS + 2u), DU = DyUnits::count(RS), XS = XUnits::sure(RS), DS = DyUnits::sure(RS);
  constexpr uint32_t tail_per = THREADS / CI;
  constexpr int TU = (int)((RS + 2u + tail_per - 1u) / tail_per);
  __shared__ __align__(16) char lds[XB + steps_dy_bytes(CO)];
  __shared__ uint32_t nan_sums;
  char *const dyl = lds + XB;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t wo = wave % WO, wc = wave / WO;

  uint32_t group, split, cog, cig;
  if (P.by_xcd) xcd_order(P.div_groups, split, group);
  else P.div_splits.divmod(blockIdx.x, group, split);
  P.div_cig.divmod(group, cog, cig);
  const uint32_t co0 = cog * CO, ci0 = cig * CI;
  const uint32_t s_begin = (uint32_t)((uint64_t)P.total_steps * split / P.splits);
  const uint32_t steps = (uint32_t)((uint64_t)P.total_steps * (split + 1u) / P.splits) - s_begin;
  if (tid == 0u) nan_sums = 0u;

  const size_t x_plane = (size_t)P.x_H * P.x_W, dy_plane = (size_t)P.H * P.W;
  const int32_t xW = (int32_t)P.x_W, dW = (int32_t)P.W, halo = P.stacked ? 1 : 0, x_rows = (int32_t)P.x_rows;

  const XUnits xu(tid, wave);
  const DyUnits du(tid, wave);
  const uint32_t q8 = 8u * xu.q, swap = octet_swap(xu.q), tail_c = tid % CI, tail_row = tid / CI;
  const uint32_t tail_to = (U * CI + (tail_c ^ octet_swap(U))) * 16u;

  // a step: row step rs of a run (an image's column tile), whether the run's rows begin with it
  struct Step {
    uint32_t run, rs, n, tile, c0, first;
    size_t x_from, dy_from;  // the image's first channel of the group, in values
  };
  auto place = [&](Step &s) {
    uint32_t plane, ctile;
    P.div_cols.divmod(s.run, plane, ctile);
    s.c0 = ctile * TW;
    s.n = plane;
    s.tile = 0u;
    if (!P.stacked) P.div_N.divmod(plane, s.tile, s.n);
    s.x_from = ((size_t)s.n * P.Cin + ci0) * x_plane;
    s.dy_from = ((size_t)s.n * P.Cout + co0) * dy_plane;
  };
  Step last;  // the last one whose rows were asked for
  P.div_row_steps.divmod(s_begin, last.run, last.rs);
  place(last);
  last.first = 1u;
  // the step whose rows are on their way
  struct Flight {
    Step s;
    uintx4 x[XU], dy[DU];
    uint32_t tail[TU];
  } f;

  // Row r of the plane, of the group's first channel.  The tiles' addresses come from lanes: a table in memory would be waited for
  // row by row.
  const uint64_t x_tile = (uint64_t)P.x[min(lane, ADH_MAX_TILES - 1u)], dy_tile = (uint64_t)P.dy[min(lane, ADH_MAX_TILES - 1u)];
  auto of_lane = [](uint64_t v, uint32_t from) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)from), hi = (uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), (int)from);
    return (uint64_t)hi << 32 | lo;
  };
  auto x_at = [&](const Step &s, int32_t r) {
    const uint32_t t = P.div_H.div((uint32_t)r);  // (not stacked: 0)
    return (const ADH_GLOBAL uint16_t *)of_lane(x_tile, s.tile + t) + (s.x_from + ((uint32_t)r - t * P.H) * P.x_W);
  };
  auto dy_at = [&](const Step &s, uint32_t R) {
    const uint32_t t = P.div_H.div(R);
    return (const ADH_GLOBAL uint16_t *)of_lane(dy_tile, s.tile + t) + (s.dy_from + (R - t * P.H) * P.W);
  };
  // (images are below 2^31 bytes)
  auto load8 = [&](const ADH_GLOBAL uint16_t *row, uint32_t channel, int32_t Q, int32_t W) {
    return *(const ADH_GLOBAL steps_u32x4 *)(row + (channel + (uint32_t)min(max(Q, 0), W - 8)));
  };
  // Channels that do not exist are taken as the group's first: what they add to is not used.
  uint32_t x_chan[XUnits::passes], dy_chan[DyUnits::passes];
#pragma unroll
  for (uint32_t p = 0; p < XUnits::passes; ++p) x_chan[p] = ci0 + xu.channel(p) < P.Cin ? xu.channel(p) * (uint32_t)x_plane : 0u;
#pragma unroll
  for (uint32_t p = 0; p < DyUnits::passes; ++p) dy_chan[p] = co0 + du.channel(p) < P.Cout ? du.channel(p) * (uint32_t)dy_plane : 0u;
  const uint32_t tail_chan = ci0 + tail_c < P.Cin ? tail_c * (uint32_t)x_plane : 0u;
  // What some steps and waves load comes first: the compiler counts what it knows to be behind a load, and waits for the rest.
  auto load = [&]() {
    f.s = last;
    const Step &s = f.s;
    const int32_t x0 = (int32_t)(s.rs * RS) - halo + (s.first ? 0 : 2), Q0 = (int32_t)s.c0 - halo;
    const uint32_t nx = s.first ? RS + 2u : RS;
    auto load_x = [&](int j) { f.x[j] = load8(x_at(s, min(max(x0 + (int32_t)xu.row_of(j), 0), x_rows - 1)), x_chan[j % XUnits::passes], Q0 + (int32_t)q8, xW); };
    auto load_dy = [&](int j) { f.dy[j] = load8(dy_at(s, min(s.rs * RS + du.row_of(j), P.rows - 1u)), dy_chan[j % DyUnits::passes], (int32_t)(s.c0 + q8), dW); };
#pragma unroll
    for (int j = 0; j < TU; ++j) {
      const uint32_t i = (uint32_t)j * tail_per + tail_row;
      if (i < nx) {
        auto row = [&](uint32_t of_wave) { return x_at(s, min(max(x0 + (int32_t)((uint32_t)j * tail_per + wave * 64u / CI + of_wave), 0), x_rows - 1)); };
        const ADH_GLOBAL uint16_t *p = row(0u);
        if (CI < 64u && lane >= CI) p = row(1u);
        f.tail[j] = *(const ADH_GLOBAL steps_u32 *)(p + (tail_chan + (uint32_t)min(Q0 + (int32_t)TW, xW - 2)));
      }
    }
#pragma unroll
    for (int j = XS; j < XU; ++j)
      if (xu.row_of(j) < nx) load_x(j);
#pragma unroll
    for (int j = DS; j < DU; ++j)
      if (du.row_of(j) < RS) load_dy(j);
#pragma unroll
    for (int j = 0; j < XS; ++j) load_x(j);
#pragma unroll
    for (int j = 0; j < DS; ++j) load_dy(j);
  };
  // eight values in their places, or none, to p
  auto store8 = [&](char *p, uintx4 u, int32_t Q, int32_t W, bool ok) {
    uintx4 v = steps_place(u, Q, W);
    if (!ok) v = uintx4{0u, 0u, 0u, 0u};
    *reinterpret_cast<uintx4 *>(p) = v;
  };
  // slot0: ring slot of the first row; buf: the dy buffer
  auto store = [&](uint32_t slot0, uint32_t buf) {
    const Step &s = f.s;
    const int32_t x0 = (int32_t)(s.rs * RS) - halo + (s.first ? 0 : 2), Q0 = (int32_t)s.c0 - halo;
    const uint32_t nx = s.first ? RS + 2u : RS;
    auto slot_of = [&](uint32_t i) {
      const uint32_t slot = slot0 + i;
      return slot - (slot >= NR ? NR : 0u);
    };
#pragma unroll
    for (int j = 0; j < XU; ++j) {
      const uint32_t i = xu.row_of(j), c = xu.channel(j);
      if (j < XS || i < nx) {
        const int32_t r = x0 + (int32_t)i;
        store8(lds + slot_of(i) * ((U + 1u) * CI * 16u) + (xu.q * CI + (c ^ swap)) * 16u, f.x[j], Q0 + (int32_t)q8, xW, r >= 0 && r < x_rows);
      }
    }
#pragma unroll
    for (int j = 0; j < TU; ++j) {
      const uint32_t i = (uint32_t)j * tail_per + tail_row;
      if (i < nx) {
        const int32_t r = x0 + (int32_t)i, d = Q0 + (int32_t)TW - min(Q0 + (int32_t)TW, xW - 2);
        const bool none = r < 0 || r >= x_rows || d >= 2;
        *reinterpret_cast<uint32_t *>(lds + slot_of(i) * ((U + 1u) * CI * 16u) + tail_to) = none ? 0u : d == 1 ? f.tail[j] >> 16 : f.tail[j];
      }
    }
#pragma unroll
    for (int j = 0; j < DU; ++j) {
      const uint32_t i = du.row_of(j), c = du.channel(j);
      if (j < DS || i < RS)
        store8(dyl + (buf * RS + i) * (U * CO * 16u) + (du.q * CO + (c ^ swap)) * 16u, f.dy[j], (int32_t)(s.c0 + q8), dW, s.rs * RS + i < P.rows);
    }
  };
  auto advance = [&]() {
    last.first = ++last.rs == P.row_steps;
    if (last.first) {
      last.rs = 0u;
      ++last.run;
      place(last);
    }
  };

  floatx4 acc[OT][9], hi[HI ? OT : 1][HI ? 9 : 1];
#pragma unroll
  for (int ot = 0; ot < OT; ++ot)
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      acc[ot][t] = floatx4{0.f, 0.f, 0.f, 0.f};
      if constexpr (HI) hi[ot][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  uint32_t chain = P.chain;  // steps that this one still takes
  auto link = [&]() {
    if constexpr (HI) {
      if (--chain != 0u) return;
      chain = P.chain;
#pragma unroll
      for (int ot = 0; ot < OT; ++ot)
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          const floatx4 sum = hi[ot][t] + acc[ot][t];
          acc[ot][t] -= sum - hi[ot][t];
          hi[ot][t] = sum;
        }
    }
  };

  // base: ring slot of the step's first x row
  auto multiply = [&](uint32_t base, uint32_t buf) {
    constexpr int kReads = 3 * (int)KB;  // (k block, window row)
    constexpr int ABUF = OT == 4 ? 1 : 2;  // (registers)
    struct Row { uintx4 d; uintx2 e; };  // an octet, the next one's first four columns
    uintx4 a[ABUF][OT];
    Row x[2];
    // this lane group's octet of k block kb: row io of the step, octet qo of the row
    auto row_of = [&](uint32_t kb) { return U >= 4u ? kb * 4u / U : kb * (4u / U) + g / U; };
    auto octet_of = [&](uint32_t kb) { return U >= 4u ? kb * 4u % U + g : g % U; };
    auto lane_at = [&](uint32_t octet, uint32_t C, uint32_t c0) { return (octet * C + c0 + (l16 ^ octet_swap(octet))) * 16u; };
    auto read_dy = [&](uint32_t kb, uintx4 (&v)[OT]) {
      const char *p = dyl + (buf * RS + row_of(kb)) * (U * CO * 16u) + lane_at(octet_of(kb), CO, wo * OT * 16u);
#pragma unroll
      for (int ot = 0; ot < OT; ++ot) v[ot] = *reinterpret_cast<const uintx4 *>(p + ot * 256u);
    };
    auto read_x = [&](int i, Row &v) {
      uint32_t slot = base + row_of(i / 3) + (uint32_t)(i % 3);
      slot -= slot >= NR ? NR : 0u;
      const char *p = lds + slot * ((U + 1u) * CI * 16u);
      v.d = *reinterpret_cast<const uintx4 *>(p + lane_at(octet_of(i / 3), CI, wc * 16u));
      v.e = *reinterpret_cast<const uintx2 *>(p + lane_at(octet_of(i / 3) + 1u, CI, wc * 16u));
    };
    read_dy(0, a[0]);
    read_x(0, x[0]);
#pragma unroll
    for (int i = 0; i < kReads; ++i) {
      if (i + 1 < kReads) {
        if (ABUF == 2 && (i + 1) % 3 == 0) read_dy((i + 1) / 3, a[(i + 1) / 3 % ABUF]);
        read_x(i + 1, x[(i + 1) & 1]);
      }
      const int r = i % 3;
      const uintx4(&av)[OT] = a[i / 3 % ABUF];
      uintx4 d = x[i & 1].d;
      asm volatile("" : "+v"(d));  // (the compiler would read the shifted columns from LDS again, dword by dword)
      const uint32_t e = x[i & 1].e[0];
      const uintx4 w[3] = {d,
                           uintx4{__builtin_amdgcn_alignbit(d[1], d[0], 16), __builtin_amdgcn_alignbit(d[2], d[1], 16),
                                  __builtin_amdgcn_alignbit(d[3], d[2], 16), __builtin_amdgcn_alignbit(e, d[3], 16)},
                           uintx4{d[1], d[2], d[3], e}};
#pragma unroll
      for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int ot = 0; ot < OT; ++ot) acc[ot][r * 3 + b] = mfma_bf16(av[ot], w[b], acc[ot][r * 3 + b]);
      if (ABUF == 1 && i % 3 == 2 && i + 1 < kReads) read_dy((i + 1) / 3, a[0]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // A step's rows are asked for two steps ahead of their products and stored one ahead, when that step's products are on their way.
  uint32_t base = 0, next = RS + 2u, buf = 0;  // next: the slot behind the step's rows
  load();
  store(0u, 0u);
  if (steps > 1u) advance();
  load();
  lds_barrier();
  for (uint32_t k = 0; k < steps; ++k) {
    multiply(base, buf);
    __builtin_amdgcn_sched_barrier(0);
    if (k + 1u == steps) break;
    link();
    store(next, buf ^ 1u);
    base = f.s.first ? next : next + NR - 2u;
    base -= base >= NR ? NR : 0u;
    next += f.s.first ? RS + 2u : RS;
    next -= next >= NR ? NR : 0u;
    buf ^= 1u;
    if (k + 2u < steps) advance();
    load();  // (or the last step's again)
    lds_barrier();
  }

  // ---- the sums to the workspace ----
  constexpr uint32_t kWave = OT * 9u * 256u;
  float *const part = P.part + ((size_t)group * P.splits + split) * (WO * WC * kWave);
  ADH_GLOBAL float *out = (ADH_GLOBAL float *)part + (size_t)wave * kWave + lane * 4u;
  bool nan = false;
#pragma unroll
  for (int ot = 0; ot < OT; ++ot)
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      floatx4 sum = acc[ot][t];
      if constexpr (HI) {
        sum += hi[ot][t];
      }
      nan |= __builtin_isunordered(sum[0], sum[1]) || __builtin_isunordered(sum[2], sum[3]);
      *(ADH_GLOBAL floatx4_u *)(out + (ot * 9 + t) * 256) = sum;
    }
  if (nan) nan_sums = 1u;
  __syncthreads();
  if (nan_sums == 0u) return;
  // sums that are NaN once more in plain fp32, straight from memory
  for (uint32_t at = tid; at < WO * WC * kWave; at += THREADS) {
    if (part[at] == part[at]) continue;
    const uint32_t i = at & 3u, ln = at >> 2 & 63u, rest = at >> 8, tap = rest % 9u, ot = rest / 9u % OT, wt = rest / 9u / OT;
    const uint32_t co = co0 + ((wt % WO) * OT + ot) * 16u + (ln >> 4) * 4u + i, ci = ci0 + (wt / WO) * 16u + (ln & 15u);
    float sum = 0.f;
    if (co < P.Cout && ci < P.Cin)
      for (uint32_t st = s_begin; st < s_begin + steps && sum == sum; ++st) {  // (a NaN stays one)
        Step s;
        P.div_row_steps.divmod(st, s.run, s.rs);
        place(s);
        for (uint32_t R = s.rs * RS; R < min((s.rs + 1u) * RS, P.rows) && sum == sum; ++R)
          for (uint32_t Q = s.c0; Q < min(s.c0 + TW, P.W) && sum == sum; ++Q) {
            const int32_t r = (int32_t)(R + tap / 3u) - halo, c = (int32_t)(Q + tap % 3u) - halo;
            const float dyv = bf16_bits_to_f32(((const ADH_GLOBAL uint16_t *)P.dy[s.tile + P.div_H.div(R)] + ((size_t)s.n * P.Cout + co) * dy_plane + (size_t)(R - P.div_H.div(R) * P.div_H.d) * P.W)[Q]);
            float xe = 0.f;
            if (r >= 0 && r < x_rows && c >= 0 && c < xW) xe = bf16_bits_to_f32(((const ADH_GLOBAL uint16_t *)P.x[s.tile + P.div_H.div((uint32_t)r)] + ((size_t)s.n * P.Cin + ci) * x_plane + (size_t)((uint32_t)r - P.div_H.div((uint32_t)r) * P.div_H.d) * P.x_W)[c]);
            sum = __builtin_fmaf(dyv, xe, sum);
          }
      }
    part[at] = sum;
  }
}

// ---- host side ----

struct StepsPlan {
  StepsParams P;
  bool co64, ci64, hi;
  uint32_t TW, groups;
  double us;
  size_t split_bytes;  // a split's sums over all channel groups
};

// Expected time of steps_per_split steps in a row by groups * splits workgroups and of adding their sums, in us, from 158 layers of 16 to
// 512 channels timed at three to five numbers of splits each (rms error 10 %).  A step takes most of its time alone, too: what it
// waits for (its instructions one after the other, LDS) is what a second workgroup on the compute unit fills.
struct StepsCost {
  double step, more;  // a step, what each further workgroup on the compute unit adds to it
  uint32_t fit;       // workgroups on a compute unit (registers, LDS)
};
static double steps_us(const StepsCost &c, uint32_t TW, uint32_t groups, uint32_t splits, uint32_t total, size_t split_bytes) {
  const double wg = (double)groups * splits / 256.0, on = std::min(std::max(wg, 1.0), (double)c.fit);
  const double step = c.step * (1.0 + c.more * (on - 1.0)) * (TW == 8u ? 1.3 : TW == 16u ? 1.03 : 1.0);
  const double rounds = std::max(1.0, 0.8 * std::ceil(wg / c.fit) + 0.2 * wg / c.fit);
  return 8.4 + ((total + splits - 1u) / splits) * step * rounds + 0.29e-6 * (double)split_bytes * splits;
}

static bool steps_plan(const StepsWgradProblem &q, StepsPlan *plan) {
  StepsParams &P = plan->P;
  if (q.W < 8u || (uint64_t)(q.H + 2ull) * q.num_tiles >= (1ull << 30) || (uint64_t)q.W >= (1ull << 30)) return false;
  if ((uint64_t)q.Cin * q.Cout * 9u >= (1ull << 31)) return false;
  if ((uint64_t)std::max(q.Cin, q.Cout) * (q.H + 2ull) * (q.W + 2ull) * 2u >= (1ull << 31)) return false;
  P.N = q.N; P.Cin = q.Cin; P.Cout = q.Cout;
  P.stacked = q.stacked ? 1u : 0u;
  P.H = q.H; P.W = q.W;
  P.x_H = q.stacked ? q.H : q.H + 2u; P.x_W = q.stacked ? q.W : q.W + 2u;
  P.rows = q.stacked ? q.H * q.num_tiles : q.H;
  P.x_rows = q.stacked ? P.rows : P.x_H;
  P.beta = q.beta;
  const uint32_t kb = kStepBlocks;
  plan->co64 = q.Cout > 32u; plan->ci64 = q.Cin > 32u;
  const uint32_t co = plan->co64 ? 64u : 32u, ci = plan->ci64 ? 64u : 32u;
  P.ci_groups = (q.Cin + ci - 1u) / ci;
  const uint32_t groups = plan->groups = P.ci_groups * ((q.Cout + co - 1u) / co);
  const uint32_t hi_co = plan->ci64 ? 32u : co, hi_groups = P.ci_groups * ((q.Cout + hi_co - 1u) / hi_co);
  plan->split_bytes = (size_t)groups * co * ci * 9u * 4u;  // (HI: no more)
  const uint64_t planes = (uint64_t)q.N * (q.stacked ? 1u : q.num_tiles);
  static const StepsCost costs[4] = {{1.15, 0.54, 4}, {1.55, 0.33, 2}, {1.4, 0.34, 3}, {1.8, 0.11, 2}};  // [co64][ci64]
  const int tile = (plan->co64 ? 2 : 0) + (plan->ci64 ? 1 : 0);
  const StepsCost &cost = costs[tile];
  const StepsCost linked = {1.26, 0.0, 1};  // (HI: and 0.84 a link; from 25 layers, rms error 6 %)
  const double link_us = 0.84;
  // The step's shape and the number of splits: the shortest expected time, steps per split going up by a quarter.  No chain of additions
  // is of more pixels than conv3x3_bf16_wgrad.hip's, whose workgroups walk down 64 columns of images (four times as many are 1.9 times
  // as far from double precision; narrow images, whose walks multiply zeros for the most part, are 1.1 times as far at as many):
  // as many splits as there were walks, or, where so many don't run at once, linked chains (HI: 512 -> 512 channels on 4 tiles of 4 x 16, 32
  // images, 486 and 150 us, relative error 4.7e-8 and 5.7e-8, by walks 576 us and 8.8e-8; with chains as long as splits 78 us and 1.8e-7).
  // Half as many pixels where enough workgroups run at once.
  const uint64_t strips = (uint64_t)q.num_tiles * q.N * ((q.W + 63u) / 64u), rows = (strips + 255u) / 256u * q.H * (q.W > 32u ? 2u : 1u);
  const uint64_t longest = (rows + 8u) / (2u * kb);
  const uint64_t walks = std::min<uint64_t>(strips, 256u) * (q.W > 32u ? 4u : 5u) / 4u;
  double best = 1e300;
  for (uint32_t TW = 32u * kb; TW >= steps_narrowest(!plan->co64 || !plan->ci64); TW /= 2u) {
    const uint32_t RS = 32u * kb / TW, row_steps = (P.rows + RS - 1u) / RS, cols = (q.W + TW - 1u) / TW;
    const uint64_t total = planes * cols * row_steps;
    if (total >= (1ull << 31)) continue;
    const uint32_t most = std::max(1u, std::min((uint32_t)total, 256u * cost.fit / std::min(groups, 256u * cost.fit)));
    const uint64_t fit = (total + most - 1u) / most, cap = std::max<uint64_t>(1u, total / walks);
    const uint64_t least = fit <= cap ? fit : (cap + 1u) / 2u, upper = fit <= cap ? std::max(fit, std::min(total, longest)) : cap;
    for (uint64_t per = least; per <= upper; per = per < upper && upper == cap ? std::min(upper, per + 1u + per / 8u) : per + 1u + per / 4u) {
      const uint32_t splits = (uint32_t)((total + per - 1u) / per);
      const double us = steps_us(cost, TW, groups, splits, (uint32_t)total, plan->split_bytes);
      if (us >= best) {
        if (us > 2.0 * best) break;
        continue;
      }
      best = us;
      plan->hi = false;
      plan->TW = TW;
      P.splits = splits;
      P.row_steps = row_steps;
      P.cols = cols;
      P.total_steps = (uint32_t)total;
    }
    // or no more splits than run at once, as chains of as many steps
    if (fit <= cap || (!plan->co64 && !plan->ci64)) continue;  // (a single group of 32 x 32 channels has splits enough)
    const uint32_t at_once = std::max(1u, std::min((uint32_t)total, 256u * linked.fit / std::min(hi_groups, 256u * linked.fit)));
    const uint64_t per = (total + at_once - 1u) / at_once;
    const uint32_t splits = (uint32_t)((total + per - 1u) / per);
    const double us = steps_us({linked.step + link_us / (double)cap, linked.more, linked.fit}, TW, hi_groups, splits, (uint32_t)total, plan->split_bytes);
    if (TW < 16u || us >= best) continue;
    best = us;
    plan->hi = true;
    plan->TW = TW;
    P.splits = splits;
    P.row_steps = row_steps;
    P.cols = cols;
    P.total_steps = (uint32_t)total;
    P.chain = (uint32_t)cap;
  }
  if (plan->hi) plan->groups = hi_groups;
  if (best == 1e300 || (uint64_t)plan->groups * P.splits >= (1ull << 22)) return false;
  plan->us = best;
  // From half of what the XCDs' caches hold (8 x 4 MB): 240 -> 16 channels on 4 tiles of 20 x 104, 81 MB, 85 -> 59 us, 1.08 in the mean from 32 MB,
  // 1.02 from 16; smaller ones lose 1 to 4 % (up to 16 %), as the partial sums' order suits the second kernel less.
  P.by_xcd = (uint64_t)q.num_tiles * q.N * q.H * q.W * (q.Cin + q.Cout) * 2u > (16ull << 20) ? 1u : 0u;
  P.div_row_steps = FastDiv(P.row_steps); P.div_cols = FastDiv(P.cols); P.div_H = FastDiv(q.stacked ? P.H : 1u << 31); P.div_N = FastDiv(P.N);
  P.div_cig = FastDiv(P.ci_groups);
  return true;
}

size_t conv3x3_wgrad_steps_workspace(const StepsWgradProblem &q) {
  StepsPlan plan = {};
  return steps_plan(q, &plan) ? (plan.split_bytes * plan.P.splits + 255u) & ~(size_t)255u : 0u;
}

double conv3x3_wgrad_steps_us(const StepsWgradProblem &q) {
  StepsPlan plan = {};
  return steps_plan(q, &plan) ? plan.us : 0.0;
}

template <int OT, int WO, int WC, bool HI>
static void launch_steps(const StepsPlan &plan, hipStream_t st) {
  const dim3 grid(plan.groups * plan.P.splits), block(64 * WO * WC);
  switch (plan.TW) {
    case 64:
      hipLaunchKernelGGL((conv3x3_wgrad_steps_kernel<64, OT, WO, WC, HI>), grid, block, 0, st, plan.P);
      break;
    case 32: hipLaunchKernelGGL((conv3x3_wgrad_steps_kernel<32, OT, WO, WC, HI>), grid, block, 0, st, plan.P); break;
    case 16: hipLaunchKernelGGL((conv3x3_wgrad_steps_kernel<16, OT, WO, WC, HI>), grid, block, 0, st, plan.P); break;
    default:
      if constexpr (!HI && 16 * OT * WO == 64 && WC == 4) hipLaunchKernelGGL((conv3x3_wgrad_steps_kernel<8, OT, WO, WC, HI>), grid, block, 0, st, plan.P);
      break;
  }
  hipLaunchKernelGGL((wgrad_sums_kernel<9, OT, WO, WC>), dim3(plan.groups * (WO * WC * OT * 9u * 64u / 16u)), dim3(256), 0, st, static_cast<const WgradSums &>(plan.P));
}
int conv3x3_wgrad_steps(const StepsWgradProblem &q, void *workspace, size_t workspace_bytes, hipStream_t st) {
  StepsPlan plan = {};
  if (!steps_plan(q, &plan) || workspace_bytes < plan.split_bytes) return ADH_EUNIMPL;
  StepsParams &P = plan.P;
  P.splits = (uint32_t)std::min<uint64_t>(P.splits, workspace_bytes / plan.split_bytes);
  P.div_groups = FastDiv(plan.groups); P.div_splits = FastDiv(P.splits);
  for (uint32_t t = 0; t < q.num_tiles; ++t) {
    P.x[t] = q.x[t];
    P.dy[t] = q.dy[t];
  }
  P.part = reinterpret_cast<float *>(workspace);
  P.dw = q.dw;
  if (plan.hi) {
    if (plan.ci64) launch_steps<1, 2, 4, true>(plan, st);
    else launch_steps<1, 4, 2, true>(plan, st);
  } else {
    if (plan.co64) plan.ci64 ? launch_steps<4, 1, 4, false>(plan, st) : launch_steps<2, 2, 2, false>(plan, st);
    else plan.ci64 ? launch_steps<2, 1, 4, false>(plan, st) : launch_steps<1, 2, 2, false>(plan, st);
  }
  return launch_status();
}

}  // namespace adh
