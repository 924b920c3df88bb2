// Convolution of an input with very few channels (an image: one to three; the stem of a network) over halo-padded fp32 tiles,
// forward and filter gradient, on the bf16 matrix cores (split_bf16.h says how).  Windows of up to eight columns at column
// stride 1 or 2, with Cin * kh rows that fit the operands; conv_thin.hip has the other shapes.
#include "conv_thin_split.h"

#include <algorithm>

#include "split_bf16.h"

namespace adh {

constexpr uint32_t kTsThreads = 256;
constexpr uint32_t kTsFar = 0x80000000u;  // a byte offset behind every buffer's end

// the bits of the magnitude, larger than any finite number's for an infinity or a NaN
__device__ __forceinline__ uint32_t worst(uint32_t so_far, float v) {
  const uint32_t b = __float_as_uint(v) & 0x7fffffffu;
  return b > so_far ? b : so_far;
}
constexpr uint32_t kTsLimitBits = 0x7f7f8000u;  // kSplitLimit's: from here on the leading part is not finite

__device__ __forceinline__ floatx4 buffer_load4(__amdgpu_buffer_rsrc_t r, uint32_t off, int imm) {
  return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, imm, 0));
}

// ---------------------------------------------------------------------------------------------
// forward: y[co][pixel] = sum over k of w[co][k] x[k at pixel]
//
// The reduction runs over octets, one per (channel, window row): the row's taps and zeros up to eight (21 octets for 7x7 over
// three channels, six k = 32 steps with 147 of 192 products real; flattened pairs would need five, but a lane could not
// read its eight values at once).  An input row lies in LDS as the eight values FROM each output column on, 16 bytes a
// column and part, so that an operand is one aligned ds_read_b128 at any window column: the thread that brings eight
// columns has their 15 (stride 2: 22) values in registers, packs the pairs once and takes the odd shifts by v_alignbit.
//   * A workgroup of four waves owns 16 MT x (1 or 2) output channels; the filter stays in registers (4 MT x Q x 3) over all the
//     tiles of 8x32 (16 x 16; half at stride 2) pixels it walks.  Two workgroups per compute unit: one stages while the
//     other multiplies, and a tile's values are on their way in registers while the one before is multiplied.
//   * Per pair of 16-pixel units and step a wave reads 6 operands for 12 MT MFMAs.  The products below h*h have sums of their own:
//     in one sum the error against double precision was 0.82 (rectified inputs 1.12, 3x3 1.35) of the v_mfma_f32 kernel's, now 0.31 (0.37, 0.48).
// Measured (64 channels; the v_mfma_f32 kernel of conv_thin.hip before): 7x7 over 3 channels, 32 images of 4 tiles of 64x256 398 -> 261 us
// (151 TFLOP/s), 7x7 / 2 on 56x112 236 -> 115; 3x3, 16 images of 32x128 75 -> 27; one image of 14x14 36 -> 10 (37 filter values a thread
// loaded in two batches instead of one by one: 19 -> 10).  Bound by the matrix cores, busy for 150 us of the first; a wave
// waited 40 % of its time while the bias was loaded behind the stores of the units before (26 % since).
// ---------------------------------------------------------------------------------------------
constexpr uint32_t kTsPartBytes = 26624;  // one part of a tile's input; three of them twice per compute unit
constexpr uint32_t kTsBlock = 128;        // bytes of eight columns
// Where column e of a block lies in it: rows (and pairs of blocks) in turn are stored in another order, so that the writes of threads
// 128 bytes apart and the reads of 16 neighbouring columns both spread over the banks.
__device__ __forceinline__ uint32_t slot_key(uint32_t line, uint32_t block) { return (line + (block & ~1u)) & 3u; }

struct ThinSplitFwdParams {
  const float *x[ADH_MAX_TILES];
  float *y[ADH_MAX_TILES];
  const float *bias[ADH_MAX_TILES];
  const float *w;
  uint32_t N, C, M, HP, WP, OH, OW, kh, kw, sh;
  uint32_t R, KK;                        // window rows over all channels; taps over all channels
  uint32_t TR, logU, logCB, RI;          // output rows of a tile; log2 of 16-column units and 8-column blocks in a row; input rows
  uint32_t pairs, tasks, cw;             // pairs of units; (channel, input row, block) triples; waves side by side in channels
  uint32_t tiles, NRB, NCB, MG;
  float beta;
  FastDiv div_MG, div_NCB, div_NRB, div_N, div_RI, div_kh;
};

template <int MT, int Q, int SW>
__global__ __launch_bounds__(kTsThreads, 2) void conv_thin_split_fwd_kernel(const ThinSplitFwdParams P) {
  __shared__ __align__(16) char lds[3 * kTsPartBytes];
  __shared__ uint32_t not_finite[3];  // of the tile, two in turn; of the filter
  const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t wm = wave & (P.cw - 1u), wp = P.cw == 2u ? wave >> 1 : wave, pw = 4u / P.cw;
  uint32_t first, mg;
  P.div_MG.divmod(blockIdx.x, first, mg);
  const uint32_t mg0 = mg * 16u * MT * P.cw, m0 = mg0 + wm * 16u * MT, step = gridDim.x / P.MG;

  // ---- the filter
  uintx4 wreg[MT][Q][3];
  {
    float *wl = reinterpret_cast<float *>(lds);
    const uint32_t rows = min(16u * MT * P.cw, P.M - mg0), n = rows * P.KK;
    if (tid == 0u) not_finite[2] = 0u;
    constexpr int kFlight = 20;  // loads in flight: a 7x7 filter of 64 channels is 37 values a thread
    for (uint32_t e0 = tid; e0 < n; e0 += kTsThreads * kFlight) {
      float f[kFlight];
#pragma unroll
      for (int k = 0; k < kFlight; ++k) f[k] = P.w[(size_t)mg0 * P.KK + min(e0 + kTsThreads * k, n - 1u)];
#pragma unroll
      for (int k = 0; k < kFlight; ++k) wl[min(e0 + kTsThreads * k, n - 1u)] = f[k];
    }
    __syncthreads();
    uint32_t bad = 0u;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const uint32_t row = wm * 16u * MT + 16u * mt + l16, o = 4u * q + g;
        const bool ok = row < rows && o < P.R;
        const float *s = wl + (ok ? row * P.KK + o * P.kw : 0u);
        float v[8];
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) {
          const bool in = ok && e < P.kw;
          v[e] = in ? s[in ? e : 0u] : 0.f;
          bad = worst(bad, v[e]);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          uint32_t h, m, l;
          split_pair(v[2 * d], v[2 * d + 1], h, m, l);
          wreg[mt][q][0][d] = h; wreg[mt][q][1][d] = m; wreg[mt][q][2][d] = l;
        }
      }
    if (bad >= kTsLimitBits) not_finite[2] = 1u;
    __syncthreads();
  }

  // ---- what a thread stages of a tile: eight columns of one input row
  constexpr int NV = SW == 1 ? 4 : 6;  // times four values
  uint32_t t_row, t_chan;
  const uint32_t t_block = tid & ((1u << P.logCB) - 1u);
  P.div_RI.divmod(tid >> P.logCB, t_chan, t_row);
  const bool t_ok = tid < P.tasks;
  const uint32_t t_off = ((t_chan * P.HP + t_row) * P.WP + t_block * 8u * SW) * 4u;
  char *const t_lds = lds + tid * kTsBlock;
  const uint32_t t_key = slot_key(tid >> P.logCB, t_block) * 16u;
  const uint32_t image_bytes = P.C * P.HP * P.WP * 4u;
  floatx4 v[NV];
  uint32_t tile = 0, n = 0, i0 = 0, j0 = 0;
  auto place = [&](uint32_t i, uint32_t &t, uint32_t &img, uint32_t &r0, uint32_t &c0) {
    uint32_t r1, r2, cb, rb;
    P.div_NCB.divmod(i, r1, cb);
    P.div_NRB.divmod(r1, r2, rb);
    P.div_N.divmod(r2, t, img);
    r0 = rb * P.TR;
    c0 = cb << (P.logCB + 3u);
  };
  // Past the last column or row the next one's values arrive, past the image's end zeros: no output that exists uses them.
  auto load = [&](uint32_t i) {
    uint32_t t, img, r0, c0;
    place(i, t, img, r0, c0);
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(P.x[t] + (size_t)img * P.C * P.HP * P.WP), 0, (int)image_bytes, 0x00020000);
    const uint32_t off = t_ok ? t_off + (r0 * P.sh * P.WP + c0 * SW) * 4u : kTsFar;
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = buffer_load4(r, off + 16u * k, 0);
  };

  // ---- where a lane's octet of a step and its pixel lie
  const uint32_t row_pitch = kTsBlock << P.logCB;
  uint32_t koff[Q];  // bytes; the line's share of the order in the low bits
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    uint32_t c, a;
    P.div_kh.divmod(4u * q + g, c, a);
    const uint32_t line = 4u * q + g < P.R ? c * P.RI + a : 0u;
    koff[q] = line * row_pitch + (line & 3u);
  }
  // the widest filter at stride 2 leaves no registers for values on their way: the other workgroup hides the wait
  constexpr bool kAhead = !(SW == 2 && MT * Q > 8);
  const bool slow_filter = not_finite[2] != 0u;
  uint32_t turn = 0u;

  if (kAhead && first < P.tiles) load(first);
  for (uint32_t i = first; i < P.tiles; i += step) {
    if (!kAhead) load(i);
    place(i, tile, n, i0, j0);
    turn ^= 1u;
    if (tid == 0u) not_finite[turn] = 0u;
    lds_barrier();  // every wave is done with the tile before
    {
      uint32_t bad = 0u;
      uint32_t d[3][2 * NV];
#pragma unroll
      for (int k = 0; k < NV; ++k) {
#pragma unroll
        for (int e = 0; e < 4; ++e) bad = worst(bad, v[k][e]);
#pragma unroll
        for (int e = 0; e < 2; ++e)
          split_pair(v[k][2 * e], v[k][2 * e + 1], d[0][2 * k + e], d[1][2 * k + e], d[2][2 * k + e]);
      }
      uint32_t key = t_key;
      asm volatile("" : "+v"(key));
      if (t_ok) {
        if (bad >= kTsLimitBits) not_finite[turn] = 1u;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            uintx4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if constexpr (SW == 2) o[e] = d[p][j + e];
              else o[e] = (j & 1) ? __builtin_amdgcn_alignbit(d[p][(j >> 1) + e + 1], d[p][(j >> 1) + e], 16) : d[p][(j >> 1) + e];
            }
            *reinterpret_cast<uintx4 *>(t_lds + p * kTsPartBytes + (j & 4) * 16 + (((j & 3) * 16) ^ key)) = o;
          }
        }
      }
    }
    lds_barrier();
    const float *const bias_t = P.bias[tile];
    float bias[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) bias[mt] = bias_t && m0 + 16u * mt + l16 < P.M ? bias_t[m0 + 16u * mt + l16] : 0.f;
    if (kAhead && i + step < P.tiles) load(i + step);
    float *const y = P.y[tile] + (size_t)n * P.M * P.OH * P.OW;
    if (slow_filter || not_finite[turn] != 0u) {
      // values whose parts are not finite: plain fp32
      const float *x = P.x[tile] + (size_t)n * P.C * P.HP * P.WP;
      const uint32_t px = P.pairs * 32u, rows = min(16u * MT * P.cw, P.M - mg0);
      for (uint32_t e = tid; e < px * rows; e += kTsThreads) {
        const uint32_t m = mg0 + e / px, u = (e % px) >> 4;
        const uint32_t row = i0 + (u >> P.logU), col = j0 + ((u & ((1u << P.logU) - 1u)) << 4) + (e & 15u);
        if (row >= P.OH || col >= P.OW) continue;
        float s = 0.f;
        for (uint32_t o = 0; o < P.R; ++o) {
          const uint32_t c = o / P.kh, a = o - c * P.kh;
          for (uint32_t b = 0; b < P.kw; ++b)
            s = fmaf(x[((size_t)c * P.HP + row * P.sh + a) * P.WP + col * SW + b], P.w[(size_t)m * P.KK + o * P.kw + b], s);
        }
        float *o = y + ((size_t)m * P.OH + row) * P.OW + col;
        if (P.beta != 0.f) s += *o;
        if (bias_t) s += bias_t[m];
        *o = s;
      }
      continue;
    }
    // a pair of units: its sums (false: below the last row), and their way out
    uint32_t row[2], col[2];
    floatx4 acc[2][MT];  // h*h of the parts; the small products have sums of their own, whose additions cost no digit of these
    auto sum = [&](uint32_t pi) {
      uint32_t at[2], key[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const uint32_t unit = 2u * pi + u, r = unit >> P.logU, cu = unit & ((1u << P.logU) - 1u);
        row[u] = i0 + r;
        col[u] = j0 + 16u * cu;
        at[u] = r * P.sh * row_pitch + cu * (2u * kTsBlock);
        key[u] = r * P.sh + 2u * cu;
      }
      if (pi >= P.pairs || row[0] >= P.OH) return false;
      floatx4 low[2][MT];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[u][mt] = low[u][mt] = floatx4{0.f, 0.f, 0.f, 0.f};
      uint32_t zero = 0u;  // (opaque: an address per step, worked out once for all tiles, is more registers than there are)
      asm volatile("" : "+v"(zero));
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        uintx4 b[2][3];
        constexpr int xp[6] = {0, 1, 2, 0, 1, 0}, wpt[6] = {2, 1, 0, 1, 0, 0};
        auto read = [&](int u) {
          const uint32_t k = koff[q] + zero;
          const char *p = lds + at[u] + (k & ~3u) + ((l16 ^ ((k + key[u]) & 3u)) << 4);
#pragma unroll
          for (int e = 0; e < 3; ++e) b[u][e] = *reinterpret_cast<const uintx4 *>(p + e * kTsPartBytes);
        };
        read(0);
        read(1);
#pragma unroll
        for (int k = 0; k < 6; ++k)
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              floatx4 &to = k < 5 ? low[u][mt] : acc[u][mt];
              to = mfma_bf16(b[u][xp[k]], wreg[mt][q][wpt[k]], to);
            }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[u][mt] += low[u][mt];
      return true;
    };
    // a lane holds pixels 4 g .. 4 g + 3 of each unit for channel l16 of each channel tile
    auto store = [&]() {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const uint32_t m = m0 + 16u * mt + l16;
        if (m >= P.M) continue;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint32_t c = col[u] + 4u * g;
          if (row[u] >= P.OH || c >= P.OW) continue;
          float *o = y + ((size_t)m * P.OH + row[u]) * P.OW + c;
          floatx4 r = acc[u][mt];
          if (c + 3u < P.OW) {
            if (P.beta != 0.f) r += *reinterpret_cast<const floatx4_u *>(o);
            if (bias_t) r += bias[mt];
            *reinterpret_cast<floatx4_u *>(o) = r;
          } else {
#pragma unroll
            for (uint32_t k = 0; k < 3u; ++k)
              if (c + k < P.OW) {
                float e = P.beta != 0.f ? o[k] + r[k] : r[k];
                if (bias_t) e += bias[mt];
                o[k] = e;
              }
          }
        }
      }
    };
    // Memory operations of a wave complete in order: the bias and the next tile's values are waited for before the first of this
    // tile's stores, not behind them.
    bool have = sum(wp);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(bias[mt]));
    if constexpr (kAhead) {
#pragma unroll
      for (int k = 0; k < NV; ++k) asm volatile("" : "+v"(v[k]));
    }
    if (have) store();
    for (uint32_t pi = wp + pw; pi < P.pairs && sum(pi); pi += pw) store();
  }
}

static bool thin_split_takes(const ThinProblem &q) {
  if (q.Cin == 0 || q.Cin > 3u || q.kw > 8u || q.sw == 0 || q.sw > 2u || q.sh == 0 || q.N == 0 || q.Cout == 0) return false;
  if ((uint64_t)q.Cin * q.HP * q.WP * 4u >= (1ull << 31) || (uint64_t)q.Cout * q.OH * q.OW * 4u >= (1ull << 31)) return false;
  return true;
}
// rows of 16 or of 32 columns, whichever covers the width with less
static uint32_t thin_split_columns(uint32_t OW) { return (OW + 15u) / 16u * 16u < (OW + 31u) / 32u * 32u ? 16u : 32u; }

int conv_thin_split_fwd(const ThinProblem &q, const void *w, void *const *y_tiles, float beta, const float *const *bias_tiles,
                        hipStream_t st) {
  if (!thin_split_takes(q) || q.Cin * q.kh > 24u) return ADH_EUNIMPL;
  ThinSplitFwdParams P = {};
  for (uint32_t t = 0; t < q.num_tiles; ++t) {
    P.x[t] = reinterpret_cast<const float *>(q.x[t]);
    P.y[t] = reinterpret_cast<float *>(y_tiles[t]);
    P.bias[t] = bias_tiles ? bias_tiles[t] : nullptr;
    if (!aligned_to(q.x[t], 4) || !aligned_to(y_tiles[t], 4)) return ADH_EUNIMPL;
  }
  P.w = reinterpret_cast<const float *>(w);
  P.N = q.N; P.C = q.Cin; P.M = q.Cout; P.HP = q.HP; P.WP = q.WP; P.OH = q.OH; P.OW = q.OW; P.kh = q.kh; P.kw = q.kw; P.sh = q.sh;
  P.R = q.Cin * q.kh;
  P.KK = P.R * q.kw;
  P.beta = beta;
  const uint32_t TW = thin_split_columns(q.OW);
  P.logU = TW == 32u ? 1u : 0u;
  P.logCB = P.logU + 1u;
  const int MT = q.Cout <= 16u ? 1 : 2;
  P.cw = q.Cout <= 32u ? 1u : 2u;
  P.MG = (q.Cout + 16u * MT * P.cw - 1u) / (16u * MT * P.cw);
  P.NCB = (q.OW + TW - 1u) / TW;
  // 256 pixels a tile; fewer where their input does not fit, and where the tiles would not go round the compute units (down
  // to a pair of units for each wave)
  uint64_t tiles = 0;
  for (P.TR = 256u / TW;; P.TR /= 2u) {
    P.RI = (P.TR - 1u) * q.sh + q.kh;
    P.tasks = q.Cin * P.RI << P.logCB;
    P.pairs = P.TR * TW / 32u;
    P.NRB = (q.OH + P.TR - 1u) / P.TR;
    tiles = (uint64_t)q.num_tiles * q.N * P.NRB * P.NCB;
    const bool fits = P.tasks <= kTsThreads && P.tasks * kTsBlock <= kTsPartBytes;
    if (fits && (tiles * P.MG >= 256u || P.pairs * P.cw <= 4u)) break;
    if (P.TR == 1u || P.TR * TW == 32u) {
      if (!fits) return ADH_EUNIMPL;
      break;
    }
  }
  if (tiles == 0 || tiles >= (1ull << 30)) return ADH_EUNIMPL;
  P.tiles = (uint32_t)tiles;
  P.div_MG = FastDiv(P.MG); P.div_NCB = FastDiv(P.NCB); P.div_NRB = FastDiv(P.NRB); P.div_N = FastDiv(q.N);
  P.div_RI = FastDiv(P.RI); P.div_kh = FastDiv(q.kh);
  // as many workgroups as stay resident, each with the same number of tiles (one more for some)
  const uint32_t most = std::max(1u, 512u / P.MG), rounds = (P.tiles + most - 1u) / most;
  const dim3 grid((P.tiles + rounds - 1u) / rounds * P.MG), block(kTsThreads);
  const uint32_t steps = (P.R + 3u) / 4u;
#define ADH_THIN(MT_, Q_, SW_) hipLaunchKernelGGL((conv_thin_split_fwd_kernel<MT_, Q_, SW_>), grid, block, 0, st, P)
#define ADH_THIN_Q(MT_, SW_)                                                                     \
  do {                                                                                           \
    if (steps <= 2u) ADH_THIN(MT_, 2, SW_);                                                      \
    else if (steps <= 4u) ADH_THIN(MT_, 4, SW_);                                                 \
    else ADH_THIN(MT_, 6, SW_);                                                                  \
  } while (0)
  if (MT == 1 && q.sw == 1u) ADH_THIN_Q(1, 1);
  else if (MT == 1) ADH_THIN_Q(1, 2);
  else if (q.sw == 1u) ADH_THIN_Q(2, 1);
  else ADH_THIN_Q(2, 2);
#undef ADH_THIN_Q
#undef ADH_THIN
  return launch_status();
}

// ---------------------------------------------------------------------------------------------
// filter gradient: dw[co][row][b] = sum over pixels of dy[co][pixel] x[row][pixel * stride + b]
//
// The reduction runs over pixels, k = 32: four octets of neighbouring output columns.  An output tile is 16 output channels
// x 16 (channel, window row) pairs for ONE window column b, so that an operand of x is an octet of its row shifted by b
// columns, the same shift for every lane: x lies in LDS as it does in memory, split (at stride 2 even and odd columns
// apart), and two aligned ds_read_b128 give the operands of every b, the odd shifts by v_alignbit (14 tiles for 7x7 over
// three channels where the flattened pairs would fill ten; those would need the eight-fold copy that forward makes).  dy goes
// from memory into the wave's registers in operand order and is split there: it is read once and never staged.
//   * A workgroup of four waves owns 16 MT x (1 or 2) output channels, all pairs and a run of tiles of 256 (stride 2: 128) pixels;
//     the waves of a channel group share the pixels.  Two workgroups per compute unit.
//   * Per 32 pixels a wave issues 12 MT NB KW/2 MFMAs against 6 NB operand reads, 2 MT loads of dy and (at stride 1)
//     36 NB shifts.
// Measured (as above): 453 -> 269 us (147 TFLOP/s), 222 -> 126, 79 -> 25, 35 -> 9.  Bound by the matrix cores, busy 64 % of the time,
// and the splitting and the shifts beside them.
// ---------------------------------------------------------------------------------------------
constexpr uint32_t kTsWgLds = 65536;

struct ThinSplitWgradParams {
  const float *x[ADH_MAX_TILES];
  const float *dy[ADH_MAX_TILES];
  float *part;  // [split][co][k]
  uint32_t N, C, M, HP, WP, OH, OW, kh, sh;
  uint32_t R, KK;
  uint32_t TR, TW, logCB, XB, RI, pitch;  // tile; log2 of octets in a row; blocks of x columns; input rows; bytes of an LDS row
  uint32_t parity_bytes, part_bytes, buffer_bytes;
  uint32_t ksteps, tasks, cw;
  uint32_t tiles, splits, NRB, NCB, MG;
  FastDiv div_MG, div_NCB, div_NRB, div_N, div_RI, div_XB, div_kh;
};

template <int MT, int NB, int KW, int SW>
__global__ __launch_bounds__(kTsThreads, 2) void conv_thin_split_wgrad_kernel(const ThinSplitWgradParams P) {
  __shared__ __align__(16) char lds[kTsWgLds];
  __shared__ uint32_t not_finite;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, l16 = lane & 15u, g = lane >> 4;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t wm = wave & (P.cw - 1u), wp = P.cw == 2u ? wave >> 1 : wave, pw = 4u / P.cw;
  uint32_t split, mg;
  P.div_MG.divmod(blockIdx.x, split, mg);
  const uint32_t mg0 = mg * 16u * MT * P.cw, m0 = mg0 + wm * 16u * MT;
  const uint32_t lo = (uint32_t)((uint64_t)P.tiles * split / P.splits), hi = (uint32_t)((uint64_t)P.tiles * (split + 1u) / P.splits);
  if (tid == 0u) not_finite = 0u;
  __syncthreads();

  auto place = [&](uint32_t i, uint32_t &t, uint32_t &img, uint32_t &r0, uint32_t &c0) {
    uint32_t r1, r2, cb, rb;
    P.div_NCB.divmod(i, r1, cb);
    P.div_NRB.divmod(r1, r2, rb);
    P.div_N.divmod(r2, t, img);
    r0 = rb * P.TR;
    c0 = cb * P.TW;
  };

  // ---- x: a thread brings 8 SW neighbouring values of one input row
  uint32_t t_line, t_block, t_chan, t_row;
  P.div_XB.divmod(tid, t_line, t_block);
  P.div_RI.divmod(t_line, t_chan, t_row);
  const bool t_ok = tid < P.tasks;
  const uint32_t t_off = ((t_chan * P.HP + t_row) * P.WP + t_block * 8u * SW) * 4u;
  const uint32_t t_lds = t_line * P.pitch + t_block * 16u;
  const uint32_t image_bytes = P.C * P.HP * P.WP * 4u;
  floatx4 xv[2 * SW];
  auto load_x = [&](uint32_t i) {
    uint32_t t, img, r0, c0;
    place(i, t, img, r0, c0);
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(P.x[t] + (size_t)img * P.C * P.HP * P.WP), 0, (int)image_bytes, 0x00020000);
    const uint32_t off = t_ok ? t_off + (r0 * P.sh * P.WP + c0 * SW) * 4u : kTsFar;
#pragma unroll
    for (int k = 0; k < 2 * SW; ++k) xv[k] = buffer_load4(r, off + 16u * k, 0);
  };
  uint32_t x_worst = 0u;
  auto store_x = [&](char *buf) {
    if (!t_ok) return;
#pragma unroll
    for (int k = 0; k < 2 * SW; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) x_worst = worst(x_worst, xv[k][e]);
#pragma unroll
    for (int s = 0; s < SW; ++s) {
      uintx4 o[3];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        // values 2 d and 2 d + 1 of this parity
        const int e0 = 2 * d * SW + s, e1 = e0 + SW;
        uint32_t h, m, l;
        split_pair(xv[e0 >> 2][e0 & 3], xv[e1 >> 2][e1 & 3], h, m, l);
        o[0][d] = h; o[1][d] = m; o[2][d] = l;
      }
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<uintx4 *>(buf + t_lds + s * P.parity_bytes + p * P.part_bytes) = o[p];
    }
  };

  // ---- dy: the lane's octet of a step for its channel of each channel tile
  const uint32_t dy_bytes = P.M * P.OH * P.OW * 4u;
  floatx4 yv[MT][2];
  int32_t y_left = 8;  // columns of the octet that exist
  auto load_dy = [&](uint32_t i, uint32_t ks) {
    uint32_t t, img, r0, c0;
    place(i, t, img, r0, c0);
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(P.dy[t] + (size_t)img * P.M * P.OH * P.OW), 0, (int)dy_bytes, 0x00020000);
    const uint32_t oct = 4u * ks + g, row = r0 + (oct >> P.logCB), col = c0 + ((oct & ((1u << P.logCB) - 1u)) << 3);
    y_left = row < P.OH ? (int32_t)P.OW - (int32_t)col : 0;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const uint32_t m = m0 + 16u * mt + l16;
      const uint32_t off = m < P.M && y_left > 0 ? ((m * P.OH + row) * P.OW + col) * 4u : kTsFar;
      yv[mt][0] = buffer_load4(r, off, 0);
      yv[mt][1] = buffer_load4(r, off + 16u, 0);
    }
  };

  uint32_t noff[NB];  // bytes of the lane's (channel, window row) pair
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    uint32_t c, a;
    P.div_kh.divmod(16u * nb + l16, c, a);
    noff[nb] = 16u * nb + l16 < P.R ? (c * P.RI + a) * P.pitch : 0u;
  }

  floatx4 acc[MT][NB][KW];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int b = 0; b < KW; ++b) acc[mt][nb][b] = floatx4{0.f, 0.f, 0.f, 0.f};
  float y_worst = 0.f;

  if (lo < hi) {
    load_x(lo);
    load_dy(lo, wp);
  }
  uint32_t buffer = 0u;
  for (uint32_t i = lo; i < hi; ++i) {
    char *const buf = lds + buffer;
    buffer = P.buffer_bytes - buffer;
    store_x(buf);
    lds_barrier();  // (the buffer before this one is free again at the next barrier)
    if (i + 1u < hi) load_x(i + 1u);
    for (uint32_t ks = wp; ks < P.ksteps; ks += pw) {
      uintx4 a[MT][3];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int e = 0; e < 4; ++e) yv[mt][k][e] = 4 * k + e < y_left ? yv[mt][k][e] : 0.f;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const float v0 = yv[mt][d >> 1][2 * (d & 1)], v1 = yv[mt][d >> 1][2 * (d & 1) + 1];
          y_worst = max_abs(y_worst, v0, v1);
          uint32_t h, m, l;
          split_pair(v0, v1, h, m, l);
          a[mt][0][d] = h; a[mt][1][d] = m; a[mt][2][d] = l;
        }
      }
      if (ks + pw < P.ksteps) load_dy(i, ks + pw);
      else if (i + 1u < hi) load_dy(i + 1u, wp);
      const uint32_t oct = 4u * ks + g;
      const char *const at = buf + (oct >> P.logCB) * P.sh * P.pitch + ((oct & ((1u << P.logCB) - 1u)) << 4);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int s = 0; s < SW; ++s) {
          uint32_t d[3][8];
#pragma unroll
          for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              const uintx4 w = *reinterpret_cast<const uintx4 *>(at + noff[nb] + s * P.parity_bytes + p * P.part_bytes + 16 * k);
#pragma unroll
              for (int e = 0; e < 4; ++e) d[p][4 * k + e] = w[e];
            }
#pragma unroll
          for (int b = s; b < KW; b += SW) {
            const int sft = b / SW;
            uintx4 o[3];
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                o[p][e] = (sft & 1) ? __builtin_amdgcn_alignbit(d[p][(sft >> 1) + e + 1], d[p][(sft >> 1) + e], 16) : d[p][(sft >> 1) + e];
            constexpr int yp[6] = {0, 1, 2, 0, 1, 0}, xp[6] = {2, 1, 0, 1, 0, 0};
#pragma unroll
            for (int k = 0; k < 6; ++k)
#pragma unroll
              for (int mt = 0; mt < MT; ++mt) acc[mt][nb][b] = mfma_bf16(a[mt][yp[k]], o[xp[k]], acc[mt][nb][b]);
          }
        }
    }
  }
  if (x_worst >= kTsLimitBits || y_worst >= kSplitLimit) not_finite = 1u;

  // ---- the sums of the waves that shared the pixels, through LDS
  floatx4 *const sums = reinterpret_cast<floatx4 *>(lds) + wm * (MT * NB * KW * 64) + lane;
  for (uint32_t w = 1; w < pw; ++w) {
    __syncthreads();
    if (wp == w) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int b = 0; b < KW; ++b) sums[((mt * NB + nb) * KW + b) * 64] = acc[mt][nb][b];
    }
    __syncthreads();
    if (wp == 0u) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int b = 0; b < KW; ++b) acc[mt][nb][b] += sums[((mt * NB + nb) * KW + b) * 64];
    }
  }
  float *const part = P.part + (size_t)split * P.M * P.KK;
  if (not_finite != 0u) {
    // values whose parts are not finite: the run's sums in plain fp32
    const uint32_t rows = min(16u * MT * P.cw, P.M - mg0);
    for (uint32_t e = tid; e < rows * P.KK; e += kTsThreads) {
      const uint32_t m = mg0 + e / P.KK, k = e % P.KK, rw = k / KW, b = k - rw * KW, c = rw / P.kh, a = rw - c * P.kh;
      float s = 0.f;
      for (uint32_t i = lo; i < hi; ++i) {
        uint32_t t, img, r0, c0;
        place(i, t, img, r0, c0);
        const float *x = P.x[t] + ((size_t)img * P.C + c) * P.HP * P.WP;
        const float *dy = P.dy[t] + ((size_t)img * P.M + m) * P.OH * P.OW;
        for (uint32_t r = r0; r < min(r0 + P.TR, P.OH); ++r)
          for (uint32_t q = c0; q < min(c0 + P.TW, P.OW); ++q)
            s = fmaf(dy[(size_t)r * P.OW + q], x[(size_t)(r * P.sh + a) * P.WP + q * SW + b], s);
      }
      part[(size_t)m * P.KK + k] = s;
    }
    return;
  }
  if (wp != 0u) return;
  // the lane holds output channels 4 g .. 4 g + 3 of a channel tile for pair l16 of a tile of pairs
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const uint32_t rw = 16u * nb + l16;
      if (rw >= P.R) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t m = m0 + 16u * mt + 4u * g + r;
        if (m >= P.M) continue;
#pragma unroll
        for (int b = 0; b < KW; ++b) part[(size_t)m * P.KK + rw * KW + b] = acc[mt][nb][b][r];
      }
    }
}

int split_sum_launch(const float *part, float *dw, uint32_t elems, uint32_t nsplit, float beta, hipStream_t st);

static bool thin_split_wgrad_plan(const ThinProblem &q, ThinSplitWgradParams *P) {
  if (!thin_split_takes(q) || q.OH == 0 || q.OW == 0) return false;
  if (q.kw != 3u && q.kw != 5u && q.kw != 7u) return false;
  if (q.Cin * q.kh > (q.kw == 7u ? 32u : 16u)) return false;
  P->N = q.N; P->C = q.Cin; P->M = q.Cout; P->HP = q.HP; P->WP = q.WP; P->OH = q.OH; P->OW = q.OW; P->kh = q.kh; P->sh = q.sh;
  P->R = q.Cin * q.kh;
  P->KK = P->R * q.kw;
  P->TW = thin_split_columns(q.OW);
  P->logCB = P->TW == 32u ? 2u : 1u;
  P->XB = P->TW / 8u + 1u;
  P->pitch = P->XB * 16u;
  P->cw = q.Cout <= 32u ? 1u : 2u;
  const uint32_t co = q.Cout <= 16u ? 16u : 32u * P->cw;
  P->MG = (q.Cout + co - 1u) / co;
  P->NCB = (q.OW + P->TW - 1u) / P->TW;
  // tiles as in forward, down to 32 pixels for each wave of a channel group
  uint64_t tiles = 0;
  for (P->TR = 256u / P->TW;; P->TR /= 2u) {
    P->RI = (P->TR - 1u) * q.sh + q.kh;
    P->tasks = q.Cin * P->RI * P->XB;
    P->parity_bytes = q.Cin * P->RI * P->pitch;
    P->part_bytes = P->parity_bytes * q.sw;
    P->buffer_bytes = 3u * P->part_bytes;
    P->ksteps = P->TR * P->TW / 32u;
    P->NRB = (q.OH + P->TR - 1u) / P->TR;
    tiles = (uint64_t)q.num_tiles * q.N * P->NRB * P->NCB;
    const bool fits = P->tasks <= kTsThreads && 2u * P->buffer_bytes <= kTsWgLds;
    if (fits && (tiles * P->MG >= 256u || P->ksteps * P->cw <= 4u)) break;
    if (P->TR * P->TW == 32u) {
      if (!fits) return false;
      break;
    }
  }
  if (tiles >= (1ull << 30)) return false;
  P->tiles = (uint32_t)tiles;
  // As many workgroups as stay resident, of four tiles or more: a workgroup's sums, written and added up, cost what a tile does
  // (64 channels, 7x7 / 2, 16 images of 56x112: 32 us with 224 workgroups, 38 with 512); a short sum over up to 128 of them.
  P->splits = std::max(1u, std::min({P->tiles, 512u / P->MG, std::max((P->tiles + 3u) / 4u, 128u / P->MG)}));
  P->div_MG = FastDiv(P->MG); P->div_NCB = FastDiv(P->NCB); P->div_NRB = FastDiv(P->NRB); P->div_N = FastDiv(q.N);
  P->div_RI = FastDiv(P->RI); P->div_XB = FastDiv(P->XB); P->div_kh = FastDiv(q.kh);
  return true;
}

size_t conv_thin_split_wgrad_workspace(const ThinProblem &q) {
  ThinSplitWgradParams P;
  if (!thin_split_wgrad_plan(q, &P)) return 0;
  return (size_t)P.splits * P.M * P.KK * sizeof(float);
}

int conv_thin_split_wgrad(const ThinProblem &q, const void *const *dy_tiles, float *dw, float beta, void *workspace,
                          size_t workspace_bytes, hipStream_t st) {
  ThinSplitWgradParams P = {};
  if (!thin_split_wgrad_plan(q, &P)) return ADH_EUNIMPL;
  P.splits = (uint32_t)std::min<uint64_t>(P.splits, workspace_bytes / ((uint64_t)P.M * P.KK * sizeof(float)));
  if (P.splits == 0u) return ADH_EUNIMPL;
  for (uint32_t t = 0; t < q.num_tiles; ++t) {
    if (!aligned_to(q.x[t], 4) || !aligned_to(dy_tiles[t], 4)) return ADH_EUNIMPL;
    P.x[t] = reinterpret_cast<const float *>(q.x[t]);
    P.dy[t] = reinterpret_cast<const float *>(dy_tiles[t]);
  }
  P.part = reinterpret_cast<float *>(workspace);
  const dim3 grid(P.splits * P.MG), block(kTsThreads);
  const bool two = P.R > 16u;
#define ADH_THIN(MT_, NB_, KW_, SW_) hipLaunchKernelGGL((conv_thin_split_wgrad_kernel<MT_, NB_, KW_, SW_>), grid, block, 0, st, P)
#define ADH_THIN_K(MT_, SW_)                                                                     \
  do {                                                                                           \
    if (q.kw == 3u) ADH_THIN(MT_, 1, 3, SW_);                                                    \
    else if (q.kw == 5u) ADH_THIN(MT_, 1, 5, SW_);                                               \
    else if (!two) ADH_THIN(MT_, 1, 7, SW_);                                                     \
    else ADH_THIN(MT_, 2, 7, SW_);                                                               \
  } while (0)
  if (q.Cout <= 16u && q.sw == 1u) ADH_THIN_K(1, 1);
  else if (q.Cout <= 16u) ADH_THIN_K(1, 2);
  else if (q.sw == 1u) ADH_THIN_K(2, 1);
  else ADH_THIN_K(2, 2);
#undef ADH_THIN_K
#undef ADH_THIN
  const int e = launch_status();
  if (e) return e;
  return split_sum_launch(P.part, dw, P.M * P.KK, P.splits, beta, st);
}

}  // namespace adh
