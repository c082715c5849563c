// The rotary rotation of a 16-byte chunk (reference arithmetic:
// ironcore/layers/positional_embedding/rotary.py:69-83), for the append kernel,
// which stores rotated rows, and the prefill kernels, which rotate query rows on
// their way into registers.
#pragma once

#include "ic_device.h"

namespace ic {

// Products and sums rounded one by one, as a sequence of separate torch ops
// is.  Contraction is off for these operations: by default the compiler may
// fuse a product into the following sum (one rounding instead of two), and
// for fp16 inputs also the widening and the final narrowing.
__device__ __forceinline__ void rotate_pair(float x1, float x2, float c, float s, float &o1, float &o2) {
#pragma clang fp contract(off)
  const float a = x1 * c;
  const float b = x2 * s;
  const float d = x1 * s;
  const float e = x2 * c;
  o1 = a - b;
  o2 = d + e;
}

template <class E>
__device__ __forceinline__ Vec16 rotate_chunk(const Vec16 &x, const float *cs, const float *sn);

template <>
__device__ __forceinline__ Vec16 rotate_chunk<F32>(const Vec16 &x, const float *cs, const float *sn) {
  const float2 c = *reinterpret_cast<const float2 *>(cs);
  const float2 s = *reinterpret_cast<const float2 *>(sn);
  float o[4];
  rotate_pair(__builtin_bit_cast(float, x.w[0]), __builtin_bit_cast(float, x.w[1]), c.x, s.x, o[0], o[1]);
  rotate_pair(__builtin_bit_cast(float, x.w[2]), __builtin_bit_cast(float, x.w[3]), c.y, s.y, o[2], o[3]);
  Vec16 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r.w[i] = __builtin_bit_cast(uint32_t, o[i]);
  return r;
}

template <class E>
__device__ __forceinline__ Vec16 rotate_chunk16(const Vec16 &x, const float *cs, const float *sn) {
  using T = typename E::type;
  const float4 c = *reinterpret_cast<const float4 *>(cs);
  const float4 s = *reinterpret_cast<const float4 *>(sn);
  const float cc[4] = {c.x, c.y, c.z, c.w};
  const float ss[4] = {s.x, s.y, s.z, s.w};
  float f[8];
  E::widen(x, f);
  Vec16 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float o1, o2;
    rotate_pair(f[2 * i], f[2 * i + 1], cc[i], ss[i], o1, o2);
    const T lo = E::narrow(o1), hi = E::narrow(o2);
    r.w[i] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
  }
  return r;
}
template <>
__device__ __forceinline__ Vec16 rotate_chunk<Bf16>(const Vec16 &x, const float *cs, const float *sn) {
  return rotate_chunk16<Bf16>(x, cs, sn);
}
template <>
__device__ __forceinline__ Vec16 rotate_chunk<F16>(const Vec16 &x, const float *cs, const float *sn) {
  return rotate_chunk16<F16>(x, cs, sn);
}

}  // namespace ic
