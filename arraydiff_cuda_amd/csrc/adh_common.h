// Shared host/device helpers for the gfx950 kernels of the spatial-conv path.
#ifndef ADH_COMMON_H
#define ADH_COMMON_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "adh_capi.h"

namespace adh {

// Division of a 31-bit value by a launch-time constant with one mul_hi, one add and one
// shift (Granlund-Montgomery round-up method).  Exact for 0 <= n < 2^31.
struct FastDiv {
  uint32_t d, mul, shift;
  FastDiv() : d(1), mul(1), shift(0) {}
  explicit FastDiv(uint32_t div) : d(div ? div : 1) {
    shift = d > 1u ? 32u - (uint32_t)__builtin_clz(d - 1u) : 0u;
    mul = (uint32_t)(((1ull << 32) * ((1ull << shift) - d)) / d + 1);
  }
  __host__ __device__ __forceinline__ uint32_t div(uint32_t n) const {
#if defined(__HIP_DEVICE_COMPILE__)
    return (__umulhi(n, mul) + n) >> shift;
#else
    return (uint32_t)(((((uint64_t)n * mul) >> 32) + n) >> shift);
#endif
  }
  __host__ __device__ __forceinline__ void divmod(uint32_t n, uint32_t &q, uint32_t &r) const {
    q = div(n);
    r = n - q * d;
  }
};

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t v) {
  return __uint_as_float(((uint32_t)v) << 16);
}

// round-to-nearest-even; NaN stays a quiet NaN (one instruction; for all 2^32 floats the bits of adding 0x7fff and the last bit and
// shifting, which takes seven)
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// A thread's vector (16 bytes, or less at its type's own alignment) at element alignment.  STREAM: non-temporal, for data that the
// on-package cache would not keep anyway.  Reads of 537 MB reach 6.9 to 7.1 TB/s that way against 5.7 to 6.4, whatever the order and
// the loads in flight.
typedef uint32_t Raw16 __attribute__((ext_vector_type(4), aligned(2)));
template <bool STREAM, typename V, typename T>
__device__ __forceinline__ V load_vec(const T *p) {
  if constexpr (sizeof(V) == 16) {
    const Raw16 *q = reinterpret_cast<const Raw16 *>(p);
    Raw16 r;
    if constexpr (STREAM) r = __builtin_nontemporal_load(q);
    else r = *q;
    V v;
    __builtin_memcpy(&v, &r, 16);
    return v;
  } else {
    return *reinterpret_cast<const V *>(p);
  }
}
template <bool STREAM, typename V, typename T>
__device__ __forceinline__ void store_vec(T *p, const V &v) {
  if constexpr (sizeof(V) == 16) {
    Raw16 *q = reinterpret_cast<Raw16 *>(p);
    Raw16 r;
    __builtin_memcpy(&r, &v, 16);
    if constexpr (STREAM) __builtin_nontemporal_store(r, q);
    else *q = r;
  } else {
    *reinterpret_cast<V *>(p) = v;
  }
}

__device__ __forceinline__ float elem_add(float a, float b) { return a + b; }
__device__ __forceinline__ uint16_t elem_add(uint16_t a, uint16_t b) {
  return f32_to_bf16_bits(bf16_bits_to_f32(a) + bf16_bits_to_f32(b));
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

inline int launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? ADH_OK : (int)e;
}

inline bool aligned_to(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

inline size_t dtype_size(int dtype) { return dtype == ADH_BF16 ? 2 : 4; }
inline bool dtype_ok(int dtype) { return dtype == ADH_F32 || dtype == ADH_BF16; }

}  // namespace adh

#endif
