// fp32 arithmetic on the bf16 matrix cores.
//
// gfx950 multiplies bf16 sixteen times as fast as fp32 (2.5 against 0.157 PFLOP/s).  An fp32 value is the exact sum of three
// bf16 values, x = h + m + l: each is the rounding of what the ones before it leave, 8 + 8 + 8 significant bits.  Products
// of bf16 values are exact in the matrix cores and their sums are fp32.  Of the nine products of two such sums the six down
// to h*l, l*h and m*m are formed; the other three are below 2^-24 of |x*w|, less than the rounding of one fp32 product.
// The matrix core rounds its sum once per 32 terms and product, the fp32 one once per term.  Six roundings at the size of the
// sum are more than fp32's where few of the 32 terms exist, and where many are zero (rectified inputs); five of them belong
// to products that are below 2^-8 of the sixth.  The kernels therefore sum those by themselves as far as registers allow.
// Relative error against double precision over that of v_mfma_f32_16x16x4_f32 sums, uniform / rectified inputs:
// convolution 0.68 / 0.91 at full chunks of 32 channels, 0.3 - 0.5 at others, 0.3 - 0.6 at stride 2 and in the stem; the filter
// gradients, whose terms are pixels and always many, 0.6 - 0.8 / 0.8 - 1.0 with all six in one sum.
// Values to take care of: one whose leading part is not finite (an infinity, or a number within half a bf16 step of the
// largest one) has inf - inf = NaN in its parts, and a NaN times the zero of a place that does not exist is one.  The kernels
// note such values, or sums that came out as NaN, and compute what they touch over again in plain fp32 from what exists.
// Below 2^-110 a value's error is 2^-134 absolute, not relative (the smallest bf16 is 2^-133).
#ifndef ADH_SPLIT_BF16_H
#define ADH_SPLIT_BF16_H

#include "adh_common.h"

namespace adh {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Memory of the device, said out loud: addresses that come out of a table in LDS would otherwise be accessed as flat ones, whose
// loads the waits for LDS operands take in.
#define ADH_GLOBAL __attribute__((address_space(1)))
// four neighbouring values, at the alignment of one
typedef floatx4 floatx4_u __attribute__((aligned(4)));

// two values' parts, packed
__device__ __forceinline__ void split_pair(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l) {
  const floatx2 v = {a, b};
  h = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  const floatx2 r = {a - __uint_as_float(h << 16), b - __uint_as_float(h & 0xffff0000u)};
  m = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
  const floatx2 s = {r[0] - __uint_as_float(m << 16), r[1] - __uint_as_float(m & 0xffff0000u)};
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector(s, bf16x2));
}

// the largest magnitude so far; a NaN leaves it alone
__device__ __forceinline__ float max_abs(float so_far, float a, float b) {
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(so_far) : "v"(a), "v"(b));
  return so_far;
}
// magnitudes from here on round to an infinite bf16
constexpr float kSplitLimit = 3.3961775e38f;

__device__ __forceinline__ floatx4 mfma_bf16(uintx4 a, uintx4 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// A kernel's only argument, read where it is used, through the scalar cache.  What a kernel with many reads once and keeps
// runs out of scalar registers, and the compiler then keeps them in lanes of vector registers, an instruction of the vector units for
// each use: 300 to 350 of 1300 to 1640 a chunk in conv3x3_split_kernel, which has none now.  The values are not known to be invariant
// to the compiler: what is used in a loop that stores is copied first.
template <typename Params>
__device__ __forceinline__ const Params &from_memory(const Params &) {
  const __attribute__((address_space(4))) Params *p = (const __attribute__((address_space(4))) Params *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const Params *)p;
}

// barrier over LDS only: memory operations in flight stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Rows of pixels in LDS as [octet of columns][channel], 16 bytes each: an octet's channels are exchanged by this (within 16).  The
// writes of a channel's octets spread over the banks, and the reads of 16 channels of an octet (the hardware takes eight of them, 0 - 3
// and 12 - 15, with the other eight of the next octet) don't meet: 4.6 cycles a ds_read_b128, 8.4 at [channel][octet].
__device__ __forceinline__ uint32_t octet_swap(uint32_t octet) { return (octet & 3u) | ((octet & 4u) ? 12u : 0u); }

// Workgroups go to the eight XCDs in turn.  This numbering gives an XCD neighbouring splits of all groups, which share what they read.
__device__ __forceinline__ void xcd_order(const FastDiv &div_groups, uint32_t &split, uint32_t &group) {
  const uint32_t xcd = blockIdx.x & 7u, per = gridDim.x >> 3, more = gridDim.x & 7u;
  div_groups.divmod(xcd * per + min(xcd, more) + (blockIdx.x >> 3), split, group);
}

}  // namespace adh
#endif
