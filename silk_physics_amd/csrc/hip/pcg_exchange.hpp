// Pieces the persistent PCG kernels share: epoch-tagged exchange words and
// small vector helpers.
#pragma once

#include "hip/device_common.hpp"
#include "hip/kernels.hpp"

namespace silk::amd::dev {

constexpr unsigned kSpinLimit = 1u << 22;

__device__ __forceinline__ void put_word(unsigned long long* w, unsigned epoch,
                                         unsigned bits) {
  __hip_atomic_store(w, (static_cast<unsigned long long>(epoch) << 32) | bits,
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void put_f3(unsigned long long* w, unsigned epoch,
                                       f3 v) {
  put_word(w, epoch, __float_as_uint(v.x));
  put_word(w + 1, epoch, __float_as_uint(v.y));
  put_word(w + 2, epoch, __float_as_uint(v.z));
}

__device__ __forceinline__ void put_double(unsigned long long* w, unsigned epoch,
                                           double v) {
  const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(v));
  put_word(w, epoch, static_cast<unsigned>(b));
  put_word(w + 1, epoch, static_cast<unsigned>(b >> 32));
}

__device__ __forceinline__ f3 fma3(float a, f3 x, f3 y) {
  return {fmaf(a, x.x, y.x), fmaf(a, x.y, y.y), fmaf(a, x.z, y.z)};
}

// Three doubles: a coarse member's residual sum.  A sum over thousands of
// slots kept as a float would carry a rounding of its initial size, which
// near convergence exceeds the sum itself.
struct d3 {
  double x, y, z;
};

__device__ __forceinline__ double ddot3(f3 a, f3 b) {
  return static_cast<double>(a.x) * b.x + static_cast<double>(a.y) * b.y +
         static_cast<double>(a.z) * b.z;
}

// x, y, z of the 16-byte record i (one LDS read).
__device__ __forceinline__ f3 lds4(const float* base, int i) {
  const float4 v = *reinterpret_cast<const float4*>(base + 4 * i);
  return {v.x, v.y, v.z};
}

__device__ __forceinline__ void sts4(float* base, int i, f3 v) {
  base[4 * i] = v.x;
  base[4 * i + 1] = v.y;
  base[4 * i + 2] = v.z;
}

// Sum over the 32 lanes of a half-wave (sum32: fixed order).
__device__ __forceinline__ f3 half_sum(f3 v) {
  return {sum32(v.x), sum32(v.y), sum32(v.z)};
}

}  // namespace silk::amd::dev
