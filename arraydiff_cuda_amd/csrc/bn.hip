// The shard-local ops between two halo exchanges: spatial batch normalisation with tile-local batch
// statistics (every rank of the reference normalises its own tile), the rectifier and the
// residual sum.  All HBM-bound.
//
// Batch norm, training forward (three launches):
//   bn_reduce_kernel<FWD>  per (tile, channel, split of the batch): sum (x - K) and sum (x - K)^2 with
//                          K = the channel's first element, so that the sums stay small next to
//                          the variance; fp32 per thread, tree over the block
//   bn_apply_kernel        first, one thread per plane of the workgroup adds the channel's splits in double:
//                          mean, 1/sqrt(var + eps), running statistics, a = scale / sqrt(var + eps) (there
//                          is no finalize launch between the two passes); then
//                          y = a*(x - mean) + shift (the difference first: the mean may be large next
//                          to the deviation), optionally max(., 0), optionally written into the interior
//                          of a halo-padded tile whose border it zeroes (BN -> ReLU -> HaloPad in
//                          one pass over the data)
// Backward mirrors it: reduce sum dy' and sum dy'*(x - mean) (dy' = dy masked by the rectifier, dy read
// from the interior of the padded gradient tile when the forward wrote a padded tile); apply works out
// the parameter gradients and three coefficients, then dx = beta*dx + k1*dy' + k2*(x - mean) + k3.
//
// Measured, fp32, 64 channels, 32 images, 4 tiles of 64 x 256 (537 MB a tensor), before (temporal accesses, one group in
// flight, coefficients before the loads) -> now: reduce 123 -> 86 us (6.2 TB/s), backward 225 -> 165 to 190; apply 240 -> 207,
// backward 320 -> 283 (5.7 TB/s).  bf16, 100 channels, 9 images, 4 tiles of 14 x 333, both passes: 135 -> 87 (the backward apply pass
// 56 -> 34: its groups no longer end where rows do; the sums stay element by element, eight in flight).
#include "adh_common.h"

#include <algorithm>
#include <type_traits>

namespace adh {

constexpr uint32_t kBnThreads = 256;

struct BnParams {
  const void *x[ADH_MAX_TILES];
  const void *dy[ADH_MAX_TILES];
  void *out[ADH_MAX_TILES];  // y (forward) or dx (backward)
  const float *scale[ADH_MAX_TILES];
  const float *shift[ADH_MAX_TILES];
  const float *mean_in[ADH_MAX_TILES];    // backward / inference: saved or fixed mean
  const float *second_in[ADH_MAX_TILES];  // backward: saved 1/sqrt(var + eps); inference: fixed variance
  float *o0[ADH_MAX_TILES];               // forward: running mean;     backward: scale gradient
  float *o1[ADH_MAX_TILES];               // forward: running variance; backward: shift gradient
  float *o2[ADH_MAX_TILES];               // forward: saved mean
  float *o3[ADH_MAX_TILES];               // forward: saved 1/sqrt(var + eps)
  float *partial;                         // [tile][c][split][2]
  uint32_t N, C, H, W, HW, p, split, n_per_split, tiles, groups_per_plane, slots_log2, along, planes_per_pass;
  uint32_t run;  // elements that lie side by side in both tensors of a pass: the plane, or (padded gradient) a row
  float eps, beta, beta_param;  // beta: input-gradient accumulation; beta_param: parameter-gradient accumulation
  int relu;
  FastDiv div_C, div_N, div_split, div_groups, div_cols;  // div_groups: what a plane is numbered by; div_cols: row length of the index that a kernel splits into (row, column)
};

__device__ __forceinline__ float bn_ld(const float *p, size_t i) { return p[i]; }
__device__ __forceinline__ float bn_ld(const uint16_t *p, size_t i) { return bf16_bits_to_f32(p[i]); }
__device__ __forceinline__ void bn_st(float *p, size_t i, float v) { p[i] = v; }
__device__ __forceinline__ void bn_st(uint16_t *p, size_t i, float v) { p[i] = f32_to_bf16_bits(v); }

// VEC elements moved by one 16-byte access at element alignment (gfx950 takes unaligned vector accesses)
template <typename T, int VEC>
struct __attribute__((packed, aligned(sizeof(T)))) BnVec {
  T v[VEC];
};
__device__ __forceinline__ float bn_f(float v) { return v; }
__device__ __forceinline__ float bn_f(uint16_t v) { return bf16_bits_to_f32(v); }
__device__ __forceinline__ void bn_t(float &d, float v) { d = v; }
__device__ __forceinline__ void bn_t(uint16_t &d, float v) { d = f32_to_bf16_bits(v); }

__device__ __forceinline__ float2 block_sum2(float a, float b) {
  __shared__ float red[2][kBnThreads / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o);
    b += __shfl_xor(b, o);
  }
  const uint32_t wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63u) == 0) {
    red[0][wave] = a;
    red[1][wave] = b;
  }
  __syncthreads();
  float2 r;
  r.x = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
  r.y = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
  return r;
}

// grid: tiles * C * split.  BWD = false: sums of (x - K), (x - K)^2.  BWD = true: sums of dy', dy' * (x - mean)
// (dy' = dy where a*(x - mean) + shift > 0 when the rectifier was fused, else dy), dy at the interior of a tile padded by p.
// VEC > 1: H*W (and, backward, W) are whole numbers of VEC-element groups, one 16-byte access per group.
// U groups a thread are loaded before the first is added (with one, the latency of a load bounds it), and are added in the
// order of a thread that takes one at a time: what a sum rounds to decides where activations tie in a pooling window.
// (U = 1 where a split has no U groups a thread: 136 channels of 1 x 46 on 8 tiles, 3 images, 4.2 us, with 8 5.6)
template <typename T, bool BWD, int VEC, int U, bool STREAM>
__global__ __launch_bounds__(kBnThreads) void bn_reduce_kernel(const BnParams P) {
  typedef BnVec<T, VEC> Vec;
  uint32_t tc, sp, tile, c;
  P.div_split.divmod(blockIdx.x, tc, sp);
  P.div_C.divmod(tc, tile, c);
  const T *x = reinterpret_cast<const T *>(P.x[tile]);
  const T *dy = reinterpret_cast<const T *>(P.dy[tile]);
  const uint32_t n0 = sp * P.n_per_split, n1 = min(P.N, n0 + P.n_per_split);
  const uint32_t WP = P.W + 2u * P.p, HPp = P.H + 2u * P.p;
  // (forward: the channel's first element, so that the sums stay small next to the variance)
  const float mean = BWD ? P.mean_in[tile][c] : bn_ld(x, (size_t)c * P.HW);
  const float a = BWD && P.relu ? P.scale[tile][c] * P.second_in[tile][c] : 0.f;
  const float b = BWD && P.relu ? P.shift[tile][c] : 0.f;
  const uint32_t groups = P.HW / (uint32_t)VEC;
  float s1 = 0.f, s2 = 0.f;
  // the groups of the split's planes are numbered through: a plane of a few groups (a late layer's 4 x 16 tile
  // is 16 of them) would otherwise leave most of the workgroup idle for one load latency per plane
  // (P.planes_per_pass planes at a time keep the running number below 2^31: one pass but for gigantic planes)
  for (uint32_t nb = n0; nb < n1; nb += P.planes_per_pass) {
    const uint32_t items = min(P.planes_per_pass, n1 - nb) * groups;
    auto load = [&](uint32_t it, Vec &xv, Vec &dv) {
      uint32_t nr, i;
      P.div_groups.divmod(it, nr, i);
      const size_t plane = (size_t)(nb + nr) * P.C + c;
      xv = load_vec<STREAM, Vec>(x + plane * P.HW + (size_t)i * VEC);
      if (!BWD) return;
      if (P.p == 0u) {
        dv = load_vec<STREAM, Vec>(dy + plane * P.HW + (size_t)i * VEC);
      } else {
        uint32_t h, w;
        P.div_cols.divmod(i, h, w);  // groups per row
        dv = load_vec<STREAM, Vec>(dy + plane * HPp * WP + (size_t)(h + P.p) * WP + P.p + w * VEC);
      }
    };
    auto add = [&](const Vec &xv, const Vec &dv) {
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        const float xc = bn_f(xv.v[k]) - mean;
        if (BWD) {
          float d = bn_f(dv.v[k]);
          if (P.relu && !(a * xc + b > 0.f)) d = 0.f;
          s1 += d;
          s2 += d * xc;
        } else {
          s1 += xc;
          s2 += xc * xc;
        }
      }
    };
    Vec xv[U], dv[U];
    uint32_t it = threadIdx.x;
    for (; it + (U - 1u) * kBnThreads < items; it += U * kBnThreads) {
#pragma unroll
      for (int u = 0; u < U; ++u) load(it + (uint32_t)u * kBnThreads, xv[u], dv[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) add(xv[u], dv[u]);
    }
    if (it < items) {  // the rest: loaded from existing places, added where it exists
#pragma unroll
      for (int u = 0; u < U - 1; ++u) {
        const uint32_t i = it + (uint32_t)u * kBnThreads;
        load(i < items ? i : it, xv[u], dv[u]);
      }
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        if (it + (uint32_t)u * kBnThreads < items) add(xv[u], dv[u]);
    }
  }
  const float2 r = block_sum2(s1, s2);
  if (threadIdx.x == 0) {
    P.partial[(size_t)blockIdx.x * 2u] = r.x;
    P.partial[(size_t)blockIdx.x * 2u + 1u] = r.y;
  }
}

// What the numbers of one (tile, channel) are worked out from; `v`: the first of the sums that this lane adds.
struct BnCoefIn {
  float scale, shift, mean, second;
  float2 v;
};
template <typename T, int MODE>
__device__ __forceinline__ BnCoefIn bn_coef_load(const BnParams &P, uint32_t tile, uint32_t c, uint32_t lane) {
  BnCoefIn in = {P.scale[tile][c], P.shift[tile][c], 0.f, 0.f, make_float2(0.f, 0.f)};
  in.mean = MODE == 0 ? bn_ld(reinterpret_cast<const T *>(P.x[tile]), (size_t)c * P.HW) : P.mean_in[tile][c];
  if (MODE != 0) in.second = P.second_in[tile][c];
  if (MODE != 1 && lane < P.split)
    in.v = *reinterpret_cast<const float2 *>(P.partial + (((size_t)tile * P.C + c) * P.split + lane) * 2u);
  return in;
}

// The five numbers the apply pass needs for one (tile, channel), worked out by `lanes` threads of every apply workgroup
// that touches the channel (the sums of the splits are added in double, in an order that hangs on `lanes` alone, the same
// over the launch, so every workgroup gets the same bits); the first of them writes cf.  `publish`: it also writes the
// channel's statistics (forward) or parameter gradients (backward); exactly one per (tile, channel) in the grid is told to.
//   MODE 0, training forward : cf = { a = scale / sqrt(var + eps), mean, shift }
//   MODE 1, inference        : the same from the fixed statistics
//   MODE 2, backward         : cf = { k1 = a, k2, k3, mean, shift };  dx = k1 dy' + k2 (x - mean) + k3
template <typename T, int MODE>
__device__ __forceinline__ void bn_plane_coef(const BnParams &P, const BnCoefIn &in, uint32_t tile, uint32_t c, uint32_t lane,
                                              uint32_t lanes, bool publish, float *cf) {
  const float scale = in.scale, shift = in.shift, K = in.mean, saved = in.second;
  if (MODE == 1) {
    if (lane != 0u) return;
    const double invstd = 1.0 / sqrt((double)saved + (double)P.eps);
    cf[0] = (float)((double)scale * invstd);
    cf[1] = K;
    cf[2] = shift;
    return;
  }
  double s1 = (double)in.v.x, s2 = (double)in.v.y;
  for (uint32_t sp = lane + lanes; sp < P.split; sp += lanes) {
    const float2 v = *reinterpret_cast<const float2 *>(P.partial + (((size_t)tile * P.C + c) * P.split + sp) * 2u);
    s1 += (double)v.x;
    s2 += (double)v.y;
  }
  for (uint32_t o = lanes >> 1; o > 0u; o >>= 1) {
    s1 += __shfl_xor(s1, (int)o);
    s2 += __shfl_xor(s2, (int)o);
  }
  if (lane != 0u) return;
  const double m = (double)P.N * (double)P.HW;
  if (MODE == 0) {
    const double d = s1 / m, mean = (double)K + d;
    double var = s2 / m - d * d;
    if (var < 0.0) var = 0.0;
    const double invstd = 1.0 / sqrt(var + (double)P.eps);
    if (publish) {
      if (P.o0[tile]) P.o0[tile][c] = (float)mean;
      if (P.o1[tile]) P.o1[tile][c] = (float)(m > 1.0 ? var * m / (m - 1.0) : var);
      if (P.o2[tile]) P.o2[tile][c] = (float)mean;
      if (P.o3[tile]) P.o3[tile][c] = (float)invstd;
    }
    cf[0] = (float)((double)scale * invstd);
    cf[1] = (float)mean;
    cf[2] = shift;
  } else {
    const double invstd = saved;
    const double dshift = s1, dscale = s2 * invstd;  // sum dy' * (x - mean) * invstd
    if (publish) {
      P.o0[tile][c] = (float)((P.beta_param != 0.f ? (double)P.o0[tile][c] : 0.0) + dscale);
      P.o1[tile][c] = (float)((P.beta_param != 0.f ? (double)P.o1[tile][c] : 0.0) + dshift);
    }
    // dx = a * (dy' - dshift/m - xhat * dscale/m),  xhat = (x - mean) * invstd
    const double a = (double)scale * invstd;
    cf[0] = (float)a;
    cf[1] = (float)(-a * invstd * dscale / m);
    cf[2] = (float)(-a * dshift / m);
    cf[3] = K;
    cf[4] = shift;  // the rectifier's mask needs the forward output's sign
  }
}

// a thread moves U groups of VEC consecutive elements, all loads before the first store: of the packed gradient plane's runs
// (backward: P.run elements, the last group ending with the run; what it shares with the one before is left to that, so
// that dx may be x or dy), of an unpadded output plane in the same way, or of a padded one (element by element where a
// group is not inside one row).
// The loads go out before the coefficients are worked out (MODE as in bn_plane_coef; there is no separate finalize
// launch): the chain of loads, sums and a square root is as long as theirs.  What that needs is loaded before them, so
// that it does not wait for them.
// Work split (bn_apply_grid): a plane of at most 128 groups takes 1 << P.slots_log2 = 16 .. 128 threads and the workgroup's
// parts take U planes each; a larger plane takes the whole workgroup, band by band (blockIdx.y): the same group of U
// planes a thread, or (P.along, backward) U groups of one plane.
template <typename T, int MODE, int VEC, bool STREAM>
__global__ __launch_bounds__(kBnThreads) void bn_apply_kernel(const BnParams P) {
  typedef BnVec<T, VEC> Vec;
  constexpr bool BWD = MODE == 2;
  constexpr uint32_t U = 4;
  __shared__ float cf_s[U * 16][8];
  const uint32_t WP = P.W + 2u * P.p, HPp = P.H + 2u * P.p;
  const uint32_t total = HPp * WP;
  const uint32_t planes = P.tiles * P.N * P.C;
  const uint32_t parts = kBnThreads >> P.slots_log2;
  const uint32_t part = threadIdx.x >> P.slots_log2;
  const bool along = BWD && P.along;
  const uint32_t per_block = along ? 1u : U * parts;  // planes
  const uint32_t gi = blockIdx.y * (along ? U * kBnThreads : kBnThreads) + (threadIdx.x & ((1u << P.slots_log2) - 1u));  // group within a plane
  const uint32_t lanes = min(8u, kBnThreads / per_block), ci = threadIdx.x / lanes, clane = threadIdx.x - ci * lanes;
  uint32_t c_tile = 0, c_n = 0, c_c = 0;
  const bool c_live = ci < per_block && blockIdx.x * per_block + ci < planes;
  BnCoefIn coef_in;
  if (c_live) {
    uint32_t tn;
    P.div_C.divmod(blockIdx.x * per_block + ci, tn, c_c);
    P.div_N.divmod(tn, c_tile, c_n);
    coef_in = bn_coef_load<T, MODE>(P, c_tile, c_c, clane);
  }
  Vec xv[U], dv[U], old[U];
  T *out_u[U];
  bool live[U];
  uint32_t skip[U], mask = (1u << VEC) - 1u, out_off = 0;
#pragma unroll
  for (uint32_t u = 0; u < U; ++u) live[u] = false;
  if (BWD) {
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t pl = along ? blockIdx.x : (blockIdx.x * parts + part) * U + u;
      const uint32_t g = along ? gi + u * kBnThreads : gi;
      live[u] = pl < planes && g < P.groups_per_plane;
      if (!live[u]) continue;
      uint32_t tn, c, tile, n, h, w;
      P.div_C.divmod(pl, tn, c);
      P.div_N.divmod(tn, tile, n);
      P.div_cols.divmod(g, h, w);  // groups of a run
      const uint32_t at = min(w * VEC, P.run - VEC);
      skip[u] = w * VEC - at;
      const size_t plane = (size_t)n * P.C + c, off = plane * P.HW + (size_t)h * P.run + at;
      out_u[u] = reinterpret_cast<T *>(P.out[tile]) + off;
      xv[u] = load_vec<STREAM, Vec>(reinterpret_cast<const T *>(P.x[tile]) + off);
      dv[u] = load_vec<STREAM, Vec>(reinterpret_cast<const T *>(P.dy[tile]) + plane * total + (size_t)(h + P.p) * WP + P.p + at);
      if (P.beta != 0.f) old[u] = load_vec<false, Vec>(out_u[u]);
    }
  } else if (gi < P.groups_per_plane) {
    // where the group sits is the same for every plane
    uint32_t r = 0, col = 0, in_off;
    bool whole = true;
    if (P.p == 0u && total >= (uint32_t)VEC) {  // the last group ends with the plane
      in_off = out_off = min(gi * VEC, total - VEC);
    } else {
      P.div_cols.divmod(gi * VEC, r, col);
      whole = r - P.p < P.H && col >= P.p && col + VEC <= P.p + P.W;  // inside one interior row
      in_off = (r - P.p) * P.W + (col - P.p);
      out_off = gi * VEC;
      if (!whole) {
        mask = 0u;
        uint32_t rr = r, cc = col;
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          if (rr - P.p < P.H && cc - P.p < P.W) mask |= 1u << k;
          if (++cc == WP) {
            cc = 0;
            ++rr;
          }
        }
      }
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t pl = (blockIdx.x * parts + part) * U + u;
      live[u] = pl < planes;
      if (!live[u]) continue;
      skip[u] = gi * VEC - out_off;
      uint32_t tn, c, tile, n;
      P.div_C.divmod(pl, tn, c);
      P.div_N.divmod(tn, tile, n);
      const T *x = reinterpret_cast<const T *>(P.x[tile]) + ((size_t)n * P.C + c) * P.HW;
      out_u[u] = reinterpret_cast<T *>(P.out[tile]) + ((size_t)n * P.C + c) * total + out_off;
      if (whole) {
        xv[u] = load_vec<STREAM, Vec>(x + in_off);
      } else {
        uint32_t rr = r, cc = col;
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          if (mask >> k & 1u) xv[u].v[k] = x[(size_t)(rr - P.p) * P.W + (cc - P.p)];
          if (++cc == WP) {
            cc = 0;
            ++rr;
          }
        }
      }
    }
  }
  if (c_live) bn_plane_coef<T, MODE>(P, coef_in, c_tile, c_c, clane, lanes, blockIdx.y == 0u && c_n == 0u, cf_s[ci]);
  __syncthreads();
#pragma unroll
  for (uint32_t u = 0; u < U; ++u) {
    if (!live[u]) continue;
    const float *cf = cf_s[along ? 0u : part * U + u];
    Vec out;
    if (!BWD) {
      const float a = cf[0], mean = cf[1], b = cf[2];
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        float v = 0.f;
        if (mask >> k & 1u) {
          v = a * (bn_f(xv[u].v[k]) - mean) + b;
          if (P.relu) v = v > 0.f ? v : 0.f;
        }
        bn_t(out.v[k], v);
      }
    } else {
      const float k1 = cf[0], k2 = cf[1], k3 = cf[2], mean = cf[3], b = cf[4];
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        const float xc = bn_f(xv[u].v[k]) - mean;
        float d = bn_f(dv[u].v[k]);
        if (P.relu && !(k1 * xc + b > 0.f)) d = 0.f;
        float g = k1 * d + k2 * xc + k3;
        if (P.beta != 0.f) g += bn_f(old[u].v[k]);
        bn_t(out.v[k], g);
      }
    }
    if (skip[u] == 0u && (BWD || out_off + VEC <= total)) {
      store_vec<STREAM, Vec>(out_u[u], out);
    } else {
#pragma unroll
      for (int k = 0; k < VEC; ++k)
        if ((uint32_t)k >= skip[u] && (BWD || out_off + k < total)) out_u[u][k] = out.v[k];
    }
  }
}

// ---- rectifier and residual sum ----

template <typename T>
__global__ __launch_bounds__(256) void relu_fwd_kernel(uint64_t n, const T *__restrict__ x, T *__restrict__ y) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) {
    const float v = bn_ld(x, i);
    bn_st(y, i, v > 0.f ? v : 0.f);
  }
}
template <typename T>
__global__ __launch_bounds__(256) void relu_bwd_kernel(uint64_t n, const T *__restrict__ y, const T *__restrict__ dy,
                                                       T *__restrict__ dx, float beta) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) {
    float g = bn_ld(y, i) > 0.f ? bn_ld(dy, i) : 0.f;
    if (beta != 0.f) g += bn_ld(dx, i);
    bn_st(dx, i, g);
  }
}
struct SumParams {
  const void *x[ADH_MAX_TILES];
  uint32_t count;
};
template <typename T>
__global__ __launch_bounds__(256) void sum_fwd_kernel(uint64_t n, const SumParams S, T *__restrict__ y) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) {
    float v = bn_ld(reinterpret_cast<const T *>(S.x[0]), i);
    for (uint32_t k = 1; k < S.count; ++k) v += bn_ld(reinterpret_cast<const T *>(S.x[k]), i);
    bn_st(y, i, v);
  }
}

// ---- host side ----

static size_t bn_ws_bytes(uint32_t tiles, uint32_t C, uint32_t split) {
  return ((size_t)tiles * C * split * 2u + (size_t)tiles * C * 8u) * 4u;
}
static uint32_t bn_split(uint32_t tiles, uint32_t N, uint32_t C) {
  const uint64_t tc = (uint64_t)tiles * C;
  return (uint32_t)std::max<uint64_t>(1u, std::min<uint64_t>(N, (2048u + tc - 1u) / tc));
}

static int bn_common(int dtype, uint32_t num_tiles, uint32_t N, uint32_t C, uint32_t H, uint32_t W, uint32_t p,
                     void *workspace, size_t workspace_bytes, BnParams *P) {
  if (!dtype_ok(dtype)) return ADH_EINVAL;
  if (num_tiles == 0 || num_tiles > ADH_MAX_TILES) return ADH_EINVAL;
  if ((uint64_t)(H + 2ull * p) * (W + 2ull * p) >= (1ull << 31) || (uint64_t)N * C * num_tiles >= (1ull << 31)) return ADH_EINVAL;
  if (p > 4096u) return ADH_EINVAL;
  P->N = N; P->C = C; P->H = H; P->W = W; P->HW = H * W; P->p = p; P->tiles = num_tiles;
  P->split = bn_split(num_tiles, N, C);
  P->n_per_split = (N + P->split - 1u) / std::max(P->split, 1u);
  P->div_C = FastDiv(C);
  P->div_split = FastDiv(P->split);
  if (N == 0 || C == 0 || H == 0 || W == 0) return ADH_OK;
  if (!workspace) return ADH_ENULL;
  if (!aligned_to(workspace, 256)) return ADH_EALIGN;
  if (workspace_bytes < bn_ws_bytes(num_tiles, C, P->split)) return ADH_EWORKSPACE;
  P->partial = reinterpret_cast<float *>(workspace);
  return ADH_OK;
}

// sets the apply kernel's work split and returns its grid.  Four groups of one plane (along) where a plane has as many: two
// tensors read and one written at the same place of four planes 64 KB apart took 311 us, of one plane 271.
static dim3 bn_apply_grid(BnParams *P, uint32_t groups_per_plane, bool backward) {
  P->groups_per_plane = groups_per_plane;
  P->div_N = FastDiv(P->N);
  // threads per plane: the whole workgroup, or for planes of at most 128 groups the power of two that holds them
  P->slots_log2 = 8;
  if (groups_per_plane <= kBnThreads / 2u) {
    P->slots_log2 = 4;
    while ((1u << P->slots_log2) < groups_per_plane) ++P->slots_log2;
  }
  const uint32_t planes = P->tiles * P->N * P->C, along = 4u * kBnThreads;
  P->along = backward && groups_per_plane >= along && planes < (1u << 24);  // (a launch has less than 2^32 threads)
  if (P->along) return dim3(planes, (groups_per_plane + along - 1u) / along);
  const uint32_t per_block = 4u * (kBnThreads >> P->slots_log2);
  return dim3((planes + per_block - 1u) / per_block, (groups_per_plane + kBnThreads - 1u) / kBnThreads);
}

// The reduce pass numbers a plane's `rows` rows of `items` (groups of elements) through.
static void bn_items(BnParams *P, uint32_t items, uint32_t rows) {
  P->div_cols = FastDiv(items);
  P->div_groups = FastDiv(items * rows);
  P->planes_per_pass = std::max(1u, 0x7fffffffu / (items * rows));
}

// The backward apply pass: a plane is `runs` runs of `run` elements, each moved as groups of `vec`.  False: one element at a
// time, where the last groups, stored element by element, are more than an eighth of all (5.6 us against 8.9 over bf16
// planes of 22), and, at row lengths that are no whole groups, where groups would be less than a workgroup per compute unit (140 tensors:
// 1.04 to 1.17 times as long by groups, up to 1.4; from 256 workgroups on 0.92, from 512 0.82).
static bool bn_runs(BnParams *P, uint32_t run, uint32_t runs, uint32_t vec) {
  bool wide = run % vec == 0u || run >= 8u * vec;
  if (wide && P->W % vec != 0u) {
    BnParams Q = *P;
    const dim3 grid = bn_apply_grid(&Q, (run + vec - 1u) / vec * runs, true);
    wide = (uint64_t)grid.x * grid.y >= 256u;
  }
  const uint32_t groups = wide ? (run + vec - 1u) / vec : run;
  P->run = run;
  P->groups_per_plane = groups * runs;
  P->div_cols = FastDiv(groups);
  return wide;
}

// `bytes`: what a pass reads.  Non-temporal where the on-package cache (256 MB, which the results go through too) cannot keep it for the
// second pass: batch norm and pooling, both passes, 32 images, 64 channels, 4 tiles, fp32 32 x 128 (134 and 268 MB) 302 us with the line at 256 MB
// and beyond, 281 from 128 to 224, 285 at 96; bf16 64 x 256 (268 and 537 MB) 616 and 608; fp32 28 and 24 images of 64 x 128 the same.
static bool bn_stream(uint64_t bytes) { return bytes > (192ull << 20); }

template <typename T, bool BWD, int VEC, bool STREAM>
static void bn_reduce(const BnParams &P, dim3 grid, hipStream_t st) {
  constexpr int U = VEC > 1 ? 4 : 8;
  if ((uint64_t)P.n_per_split * P.div_groups.d >= (uint64_t)U * kBnThreads)
    hipLaunchKernelGGL((bn_reduce_kernel<T, BWD, VEC, U, STREAM>), grid, dim3(kBnThreads), 0, st, P);
  else
    hipLaunchKernelGGL((bn_reduce_kernel<T, BWD, VEC, 1, false>), grid, dim3(kBnThreads), 0, st, P);
}

template <typename F>
static void bn_launch(bool stream_data, int dtype, F f) {
  if (dtype == ADH_F32) {
    if (stream_data) f(std::true_type{}, 0.f);
    else f(std::false_type{}, 0.f);
  } else {
    if (stream_data) f(std::true_type{}, uint16_t(0));
    else f(std::false_type{}, uint16_t(0));
  }
}

}  // namespace adh

using namespace adh;

extern "C" {

size_t adh_batchnorm2d_workspace_bytes(uint32_t num_tiles, uint32_t N, uint32_t C) {
  if (num_tiles == 0 || num_tiles > ADH_MAX_TILES) return 0;
  return (bn_ws_bytes(num_tiles, C, bn_split(num_tiles, N, C)) + 255u) & ~(size_t)255u;
}

int adh_batchnorm2d_fwd_tiles(int dtype, int training, uint32_t num_tiles, uint32_t N, uint32_t C, uint32_t H, uint32_t W,
                              float eps, int relu, uint32_t out_halo, const void *const *x_tiles,
                              const float *const *scale_tiles, const float *const *shift_tiles,
                              const float *const *fixed_mean_tiles, const float *const *fixed_var_tiles,
                              void *const *y_tiles, float *const *run_mean_tiles, float *const *run_var_tiles,
                              float *const *save_mean_tiles, float *const *save_invstd_tiles, void *workspace,
                              size_t workspace_bytes, void *stream) {
  BnParams P = {};
  int e = bn_common(dtype, num_tiles, N, C, H, W, out_halo, workspace, workspace_bytes, &P);
  if (e) return e;
  if (N == 0 || C == 0 || H == 0 || W == 0) return ADH_OK;
  if (!(eps >= 0.f)) return ADH_EINVAL;
  if (!x_tiles || !scale_tiles || !shift_tiles || !y_tiles) return ADH_ENULL;
  if (!training && (!fixed_mean_tiles || !fixed_var_tiles)) return ADH_ENULL;
  const size_t es = dtype_size(dtype);
  for (uint32_t t = 0; t < num_tiles; ++t) {
    if (!x_tiles[t] || !scale_tiles[t] || !shift_tiles[t] || !y_tiles[t]) return ADH_ENULL;
    if (!aligned_to(x_tiles[t], es) || !aligned_to(y_tiles[t], es)) return ADH_EALIGN;
    P.x[t] = x_tiles[t];
    P.out[t] = y_tiles[t];
    P.scale[t] = scale_tiles[t];
    P.shift[t] = shift_tiles[t];
    if (training) {
      P.o0[t] = run_mean_tiles ? run_mean_tiles[t] : nullptr;
      P.o1[t] = run_var_tiles ? run_var_tiles[t] : nullptr;
      P.o2[t] = save_mean_tiles ? save_mean_tiles[t] : nullptr;
      P.o3[t] = save_invstd_tiles ? save_invstd_tiles[t] : nullptr;
    } else {
      if (!fixed_mean_tiles[t] || !fixed_var_tiles[t]) return ADH_ENULL;
      P.mean_in[t] = fixed_mean_tiles[t];
      P.second_in[t] = fixed_var_tiles[t];
    }
  }
  P.eps = eps;
  P.relu = relu ? 1 : 0;
  hipStream_t st = as_stream(stream);
  const uint32_t tc = num_tiles * C, vec = (uint32_t)(16 / es);
  const uint32_t gpp = ((H + 2u * out_halo) * (W + 2u * out_halo) + vec - 1u) / vec;
  if ((gpp + kBnThreads - 1u) / kBnThreads > 65535u) return ADH_EINVAL;  // grid.y
  const bool stream_data = bn_stream((uint64_t)tc * N * H * W * es);
  if (training) {
    const bool wide = H * W % vec == 0u;  // the statistics pass reads whole 16-byte groups
    bn_items(&P, H * W / (wide ? vec : 1u), 1u);
    bn_launch(stream_data, dtype, [&](auto s, auto t) {
      typedef decltype(t) T;
      if (wide) bn_reduce<T, false, 16 / sizeof(T), s>(P, dim3(tc * P.split), st);
      else bn_reduce<T, false, 1, false>(P, dim3(tc * P.split), st);
    });
  }
  P.div_cols = FastDiv(W + 2u * out_halo);  // the apply kernel walks the padded output plane
  const dim3 grid = bn_apply_grid(&P, gpp, false);
  bn_launch(stream_data, dtype, [&](auto s, auto t) {
    typedef decltype(t) T;
    if (training) hipLaunchKernelGGL((bn_apply_kernel<T, 0, 16 / sizeof(T), s>), grid, dim3(kBnThreads), 0, st, P);
    else hipLaunchKernelGGL((bn_apply_kernel<T, 1, 16 / sizeof(T), s>), grid, dim3(kBnThreads), 0, st, P);
  });
  return launch_status();
}

int adh_batchnorm2d_bwd_tiles(int dtype, uint32_t num_tiles, uint32_t N, uint32_t C, uint32_t H, uint32_t W, int relu,
                              uint32_t dy_halo, const void *const *x_tiles, const void *const *dy_tiles,
                              const float *const *scale_tiles, const float *const *shift_tiles,
                              const float *const *save_mean_tiles, const float *const *save_invstd_tiles,
                              void *const *dx_tiles, float *const *dscale_tiles, float *const *dshift_tiles,
                              float beta_data, float beta_param, void *workspace, size_t workspace_bytes,
                              void *stream) {
  BnParams P = {};
  int e = bn_common(dtype, num_tiles, N, C, H, W, dy_halo, workspace, workspace_bytes, &P);
  if (e) return e;
  if ((beta_data != 0.f && beta_data != 1.f) || (beta_param != 0.f && beta_param != 1.f)) return ADH_EINVAL;
  if (N == 0 || C == 0 || H == 0 || W == 0) return ADH_OK;
  if (!x_tiles || !dy_tiles || !scale_tiles || !save_mean_tiles || !save_invstd_tiles || !dx_tiles || !dscale_tiles ||
      !dshift_tiles)
    return ADH_ENULL;
  if (relu && !shift_tiles) return ADH_ENULL;
  const size_t es = dtype_size(dtype);
  for (uint32_t t = 0; t < num_tiles; ++t) {
    if (!x_tiles[t] || !dy_tiles[t] || !scale_tiles[t] || !save_mean_tiles[t] || !save_invstd_tiles[t] || !dx_tiles[t] ||
        !dscale_tiles[t] || !dshift_tiles[t] || (relu && !shift_tiles[t]))
      return ADH_ENULL;
    if (!aligned_to(x_tiles[t], es) || !aligned_to(dy_tiles[t], es) || !aligned_to(dx_tiles[t], es)) return ADH_EALIGN;
    P.x[t] = x_tiles[t];
    P.dy[t] = dy_tiles[t];
    P.out[t] = dx_tiles[t];
    P.scale[t] = scale_tiles[t];
    P.shift[t] = shift_tiles ? shift_tiles[t] : scale_tiles[t];
    P.mean_in[t] = save_mean_tiles[t];
    P.second_in[t] = save_invstd_tiles[t];
    P.o0[t] = dscale_tiles[t];
    P.o1[t] = dshift_tiles[t];
  }
  P.relu = relu ? 1 : 0;
  hipStream_t st = as_stream(stream);
  const uint32_t tc = num_tiles * C, vec = (uint32_t)(16 / es);
  const bool rwide = W % vec == 0u;  // the sums are of whole 16-byte groups of a row
  const bool awide = dy_halo ? bn_runs(&P, W, H, vec) : bn_runs(&P, H * W, 1u, vec);
  if ((P.groups_per_plane + kBnThreads - 1u) / kBnThreads > 65535u) return ADH_EINVAL;  // grid.y
  const bool stream_data = bn_stream((uint64_t)tc * N * H * W * es * 2u);
  P.beta = beta_data;
  P.beta_param = beta_param;
  const uint32_t apply_groups = P.groups_per_plane;
  const FastDiv apply_cols = P.div_cols;
  bn_items(&P, W / (rwide ? vec : 1u), H);
  const dim3 rgrid(tc * P.split);
  bn_launch(stream_data, dtype, [&](auto s, auto t) {
    typedef decltype(t) T;
    if (rwide) bn_reduce<T, true, 16 / sizeof(T), s>(P, rgrid, st);
    else bn_reduce<T, true, 1, false>(P, rgrid, st);
  });
  P.div_cols = apply_cols;
  const dim3 agrid = bn_apply_grid(&P, apply_groups, true);
  bn_launch(stream_data, dtype, [&](auto s, auto t) {
    typedef decltype(t) T;
    if (awide) hipLaunchKernelGGL((bn_apply_kernel<T, 2, 16 / sizeof(T), s>), agrid, dim3(kBnThreads), 0, st, P);
    else hipLaunchKernelGGL((bn_apply_kernel<T, 2, 1, false>), agrid, dim3(kBnThreads), 0, st, P);
  });
  return launch_status();
}

static uint32_t flat_blocks(uint64_t n) { return (uint32_t)std::min<uint64_t>((n + 1023u) / 1024u, 1u << 20); }

int adh_relu_fwd(int dtype, uint64_t n, const void *x, void *y, void *stream) {
  if (!dtype_ok(dtype)) return ADH_EINVAL;
  if (n == 0) return ADH_OK;
  if (!x || !y) return ADH_ENULL;
  if (!aligned_to(x, dtype_size(dtype)) || !aligned_to(y, dtype_size(dtype))) return ADH_EALIGN;
  if (dtype == ADH_F32)
    hipLaunchKernelGGL(relu_fwd_kernel<float>, dim3(flat_blocks(n)), dim3(256), 0, as_stream(stream), n,
                       reinterpret_cast<const float *>(x), reinterpret_cast<float *>(y));
  else
    hipLaunchKernelGGL(relu_fwd_kernel<uint16_t>, dim3(flat_blocks(n)), dim3(256), 0, as_stream(stream), n,
                       reinterpret_cast<const uint16_t *>(x), reinterpret_cast<uint16_t *>(y));
  return launch_status();
}

int adh_relu_bwd(int dtype, uint64_t n, const void *y, const void *dy, void *dx, float beta, void *stream) {
  if (!dtype_ok(dtype) || (beta != 0.f && beta != 1.f)) return ADH_EINVAL;
  if (n == 0) return ADH_OK;
  if (!y || !dy || !dx) return ADH_ENULL;
  const size_t es = dtype_size(dtype);
  if (!aligned_to(y, es) || !aligned_to(dy, es) || !aligned_to(dx, es)) return ADH_EALIGN;
  if (dtype == ADH_F32)
    hipLaunchKernelGGL(relu_bwd_kernel<float>, dim3(flat_blocks(n)), dim3(256), 0, as_stream(stream), n,
                       reinterpret_cast<const float *>(y), reinterpret_cast<const float *>(dy),
                       reinterpret_cast<float *>(dx), beta);
  else
    hipLaunchKernelGGL(relu_bwd_kernel<uint16_t>, dim3(flat_blocks(n)), dim3(256), 0, as_stream(stream), n,
                       reinterpret_cast<const uint16_t *>(y), reinterpret_cast<const uint16_t *>(dy),
                       reinterpret_cast<uint16_t *>(dx), beta);
  return launch_status();
}

int adh_sum_fwd(int dtype, uint32_t num_inputs, uint64_t n, const void *const *xs, void *y, void *stream) {
  if (!dtype_ok(dtype) || num_inputs == 0 || num_inputs > ADH_MAX_TILES) return ADH_EINVAL;
  if (n == 0) return ADH_OK;
  if (!xs || !y) return ADH_ENULL;
  const size_t es = dtype_size(dtype);
  SumParams S = {};
  S.count = num_inputs;
  for (uint32_t k = 0; k < num_inputs; ++k) {
    if (!xs[k]) return ADH_ENULL;
    if (!aligned_to(xs[k], es)) return ADH_EALIGN;
    S.x[k] = xs[k];
  }
  if (!aligned_to(y, es)) return ADH_EALIGN;
  if (dtype == ADH_F32)
    hipLaunchKernelGGL(sum_fwd_kernel<float>, dim3(flat_blocks(n)), dim3(256), 0, as_stream(stream), n, S,
                       reinterpret_cast<float *>(y));
  else
    hipLaunchKernelGGL(sum_fwd_kernel<uint16_t>, dim3(flat_blocks(n)), dim3(256), 0, as_stream(stream), n, S,
                       reinterpret_cast<uint16_t *>(y));
  return launch_status();
}

}  // extern "C"
