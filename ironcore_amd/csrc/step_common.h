// Pieces shared by the kernels of a decode step's linears (step_linear.hip, step_stack.hip): the product of a lane's block
// of W, the activations.
#pragma once

#include "ic_device.h"
#include "../../include/ironcore_paged.h"

namespace ic {
namespace step {

constexpr int kStepWaves = 8;
constexpr int kStepThreads = kStepWaves * kWave;
constexpr int kXcds = 8;

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

struct StepBf16 {
  using E = Bf16;
  static __device__ __forceinline__ f32x4_t mma(const Vec16 &a, const Vec16 &b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  }
};
struct StepF16 {
  using E = F16;
  static __device__ __forceinline__ f32x4_t mma(const Vec16 &a, const Vec16 &b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
  }
};
struct StepF32 {
  using E = F32;
};

// NW 32-bit words of a row of W.
template <int NW>
struct alignas(4 * NW) Words {
  uint32_t w[NW];
};

template <class M, int NB>
struct Shape {
  static constexpr int ES = sizeof(typename M::E::type);
  static constexpr int KR = M::E::EPL;        // rows of W in a lane's block
  static constexpr int STEP = 4 * KR;         // k of a step (64 bytes of a row of x)
  static constexpr int TN = 16 * NB;          // columns of a workgroup
  static constexpr int NW = NB * ES / 4;
  static constexpr int PITCH = TN + 4;        // of the waves' sums in LDS
  // steps in flight: 64 registers of W
  static constexpr int D = 64 / (KR * NW) > 8 ? 8 : 64 / (KR * NW);
};

// acc[j][t] += the product of a lane's block (row r of it in wv[r]) and x: matrix row c of MFMA j is column c * NB + j
// of the tile.
template <class M, int MT, int NB>
__device__ __forceinline__ void multiply(const Words<Shape<M, NB>::NW> (&wv)[Shape<M, NB>::KR], const Vec16 (&xv)[MT],
                                         f32x4_t (&acc)[NB][MT]) {
  if constexpr (Shape<M, NB>::ES == 2) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      Vec16 a;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        a.w[r] = __builtin_amdgcn_perm(wv[2 * r + 1].w[j / 2], wv[2 * r].w[j / 2], j & 1 ? 0x07060302u : 0x05040100u);
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[j][t] = M::mma(a, xv[t], acc[j][t]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, wv[r].w[j]),
                                                           __builtin_bit_cast(float, xv[t].w[r]), acc[j][t], 0, 0, 0);
  }
}

__device__ __forceinline__ float sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

__device__ __forceinline__ float activate(int act, float x) {
  switch (act) {
    case IC_ACT_RELU: return x < 0.f ? 0.f : x;
    case IC_ACT_GELU: return 0.5f * x * (1.f + erff(x * 0.70710678118654752440f));
    case IC_ACT_SILU: return x * sigmoid(x);
    default: return x;
  }
}

template <class T>
struct alignas(2 * sizeof(T)) Pair {
  T a, b;
};

}  // namespace step
}  // namespace ic
