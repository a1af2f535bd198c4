// Accumulator values published between blocks (look-back of the segmented
// walks): flagged 64-bit words, one per 32 bits of accumulator, written and read
// with relaxed agent-scope atomics; a word's flag is zero until it is published.
#pragma once

#include "em_common.h"

namespace rem {

constexpr int kWalkSpin = 1 << 20;  // bounded wait of one look-back read

template <typename Acc>
struct Pub;
template <>
struct Pub<float> {
  static constexpr int W = 1;  // 64-bit words per value: flag << 32 | bits
  static __device__ __forceinline__ void put(uint64_t* p, float v, uint32_t flag) {
    __hip_atomic_store(p, ((uint64_t)flag << 32) | __float_as_uint(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  // false while the value is not published (or the spin limit ran out)
  static __device__ __forceinline__ bool get(uint64_t* p, float* v, uint32_t* flag) {
    uint64_t w = 0;
    for (int spin = 0; spin < kWalkSpin; ++spin) {
      w = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (w >> 32) break;
      __builtin_amdgcn_s_sleep(1);
    }
    *v = __uint_as_float((uint32_t)w);
    *flag = (uint32_t)(w >> 32);
    return *flag != 0;
  }
  // the words of one value as read once (no wait), and their value when published
  static __device__ __forceinline__ void peek(uint64_t* p, uint64_t* w) {
    w[0] = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ bool decode(const uint64_t* w, float* v, uint32_t* flag) {
    *v = __uint_as_float((uint32_t)w[0]);
    *flag = (uint32_t)(w[0] >> 32);
    return *flag != 0;
  }
};
template <>
struct Pub<double> {
  static constexpr int W = 2;  // high half, low half
  static __device__ __forceinline__ void put(uint64_t* p, double v, uint32_t flag) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    Pub<float>::put(p, __uint_as_float((uint32_t)(b >> 32)), flag);
    Pub<float>::put(p + 1, __uint_as_float((uint32_t)b), flag);
  }
  static __device__ __forceinline__ bool get(uint64_t* p, double* v, uint32_t* flag) {
    float hi, lo;
    uint32_t f0, f1;
    const bool ok = Pub<float>::get(p, &hi, &f0) & Pub<float>::get(p + 1, &lo, &f1);
    *v = __longlong_as_double(
        (long long)(((uint64_t)__float_as_uint(hi) << 32) | (uint64_t)__float_as_uint(lo)));
    *flag = f0;
    return ok;
  }
  static __device__ __forceinline__ void peek(uint64_t* p, uint64_t* w) {
    w[0] = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    w[1] = __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ bool decode(const uint64_t* w, double* v, uint32_t* flag) {
    *v = __longlong_as_double((long long)((w[0] << 32) | (w[1] & 0xffffffffull)));
    *flag = (uint32_t)(w[0] >> 32);
    return (w[0] >> 32) != 0 && (w[1] >> 32) != 0;
  }
};

}  // namespace rem
