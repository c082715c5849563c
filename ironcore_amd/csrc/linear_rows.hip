// y = x W (+ bias) for a few rows of x: the projections of a decode step.
//
// The reference's linears keep W as [in, out] (ironcore/parallel/tensor_parallel/
// layers.py:41,194-204).  With at most 32 rows the product is a stream over W:
// HBM-bound, as long as enough of W is on its way and every CU takes part.
//
//  * MFMA with W as the A operand (its columns are the matrix rows) and x as B, in
//    the k order that W's layout gives: a lane loads KB rows x NB columns of W,
//    16 bytes a row, 16 lanes side by side (256 bytes of a row), and W never passes
//    through LDS.  fp32: v_mfma_f32_16x16x4 takes the values as they lie; 16 bits:
//    8 x 8 values are transposed within the lane (one v_perm per register) for
//    v_mfma_f32_16x16x32.
//  * A workgroup is 8 waves on the same 16 * NB columns; they take the k steps in
//    turn (all loads of a step and of the next one in flight) and add up through LDS.
//  * Few columns leave CUs idle, so the k range is split over workgroups, whose
//    partial sums (fp32) a second launch adds in a fixed order, with the bias.
//
// bf16, 16 rows, W from memory (time of torch's library product / of this kernel, both
// launches): 4 096 x 4 096 21.8 / 12.2 us, 11 008 x 4 096 67.3 / 21.9, 4 096 x 22 016
// 52.1 / 37.8 (4.8 TB/s), 4 096 x 32 000 53.4 / 44.4 (5.9 TB/s); fp32, 4 rows, with the
// bias: 768 x 768 9.9 / 6.9, 768 x 3 072 12.9 / 8.3, 3 072 x 768 20.7 / 7.6.  Distance to
// float64: 16 bits 1.65e-3 against 2.3e-3 with a bias (rounded once), fp32 at 4 096
// products 1.6e-7 against 5.5e-7.
#include "ic_device.h"
#include "ic_internal.h"
#include "../../include/ironcore_paged.h"

namespace ic {

namespace {

constexpr int kLinearWaves = 8;
constexpr int kLinearThreads = kLinearWaves * kWave;

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

struct LinearKP {
  const char *x, *w, *bias;
  char *out;
  float *partials;  // [splits][m][n], splits > 1
  int64_t x_stride, w_stride, out_stride;  // elements
  int m, n, steps, per_split;
};

// v_perm of two registers: the low (high) halves of a and b side by side.
__device__ __forceinline__ uint32_t low_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

struct LinearBf16 {
  using E = Bf16;
  static __device__ __forceinline__ f32x4_t mma(const Vec16 &a, const Vec16 &b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  }
};
struct LinearF16 {
  using E = F16;
  static __device__ __forceinline__ f32x4_t mma(const Vec16 &a, const Vec16 &b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
  }
};
struct LinearF32 {
  using E = F32;
};

// acc[j][t] += the product of the lane block wv (row r of it in wv[r]) and x: matrix row c of MFMA j is column
// c * NB + j of the workgroup's.
template <class M, int MT>
__device__ __forceinline__ void multiply(const Vec16 (&wv)[M::E::EPL], const Vec16 (&xv)[MT],
                                         f32x4_t (&acc)[M::E::EPL][MT]) {
  if constexpr (M::E::EPL == 8) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      Vec16 a;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        a.w[r] = j & 1 ? high_halves(wv[2 * r].w[j / 2], wv[2 * r + 1].w[j / 2])
                       : low_halves(wv[2 * r].w[j / 2], wv[2 * r + 1].w[j / 2]);
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[j][t] = M::mma(a, xv[t], acc[j][t]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, wv[r].w[j]),
                                                           __builtin_bit_cast(float, xv[t].w[r]), acc[j][t], 0, 0, 0);
  }
}

template <class M, int MT, bool SPLIT>
__global__ __launch_bounds__(kLinearThreads) void linear_rows_kernel(const LinearKP p) {
  using E = typename M::E;
  using T = typename E::type;
  constexpr int NB = E::EPL;    // columns and rows of a lane's block
  constexpr int TN = 16 * NB;   // columns of the workgroup
  constexpr int STEP = 4 * NB;  // k of a step
  constexpr int ES = sizeof(T);
  constexpr int PITCH = kWave + 1;
  __shared__ float s_acc[kLinearWaves][NB * 4 * PITCH];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int c = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * TN;
  const int col = n0 + c * NB < p.n ? n0 + c * NB : p.n - NB;  // (columns past the end: loaded, never stored)
  const int first = blockIdx.y * p.per_split;
  const int end = first + p.per_split < p.steps ? first + p.per_split : p.steps;
  const char *w = p.w + ((int64_t)g * NB * p.w_stride + col) * ES;
  const char *x[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int row = t * 16 + c < p.m ? t * 16 + c : p.m - 1;
    x[t] = p.x + (row * p.x_stride + g * NB) * ES;
  }
  f32x4_t acc[NB][MT];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[j][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  Vec16 wv[2][NB], xv[2][MT];
  auto load = [&](int step, int b) {
    const char *at = w + (int64_t)step * STEP * p.w_stride * ES;
#pragma unroll
    for (int r = 0; r < NB; ++r) wv[b][r] = load16(at + r * p.w_stride * ES);
#pragma unroll
    for (int t = 0; t < MT; ++t) xv[b][t] = load16(x[t] + (int64_t)step * STEP * ES);
  };
  // two steps a round; a step past the end loads the last one again and is left out of the sums
  const int last = end - 1;
  int step = first + wave;
  if (step < end) load(step, 0);
  for (; step < end; step += 2 * kLinearWaves) {
    const int second = step + kLinearWaves, third = second + kLinearWaves;
    load(second < end ? second : last, 1);
    multiply<M, MT>(wv[0], xv[0], acc);
    if (third < end) load(third, 0);
    if (second < end) multiply<M, MT>(wv[1], xv[1], acc);
  }
  // ---- the waves' sums, 16 rows of x at a time -------------------------------------------
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (t > 0) __syncthreads();
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) s_acc[wave][(j * 4 + i) * PITCH + lane] = acc[j][t][i];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * TN; e += kLinearThreads) {
      const int row = e / TN, at = e % TN;             // matrix row r of MFMA j is column r * NB + j
      const int j = at % NB, r = at / NB;
      const int slot = (j * 4 + (r & 3)) * PITCH + (r >> 2) * 16 + row;
      float sum = 0.f;
#pragma unroll
      for (int v = 0; v < kLinearWaves; ++v) sum += s_acc[v][slot];
      const int m = t * 16 + row, n = n0 + at;
      if (m >= p.m || n >= p.n) continue;
      if constexpr (SPLIT) {
        p.partials[((int64_t)blockIdx.y * p.m + m) * p.n + n] = sum;
      } else {
        if (p.bias != nullptr) sum += static_cast<float>(reinterpret_cast<const T *>(p.bias)[n]);
        reinterpret_cast<T *>(p.out)[m * p.out_stride + n] = E::narrow(sum);
      }
    }
  }
}

constexpr int kLinearSumThreads = 128;

// Adds the splits' partial sums in order, four columns a lane.  Bound by the round trips to them.
template <class E>
__global__ __launch_bounds__(kLinearSumThreads) void linear_rows_sum_kernel(const LinearKP p, int splits) {
  using T = typename E::type;
  const int n = (blockIdx.x * kLinearSumThreads + threadIdx.x) * 4;
  if (n >= p.n) return;
  const int m = blockIdx.y;
  const float *at = p.partials + (int64_t)m * p.n + n;
  const int64_t pitch = (int64_t)p.m * p.n;
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < splits; ++s) {
    const float4 v = *reinterpret_cast<const float4 *>(at + s * pitch);
    sum[0] += v.x, sum[1] += v.y, sum[2] += v.z, sum[3] += v.w;
  }
  T *to = reinterpret_cast<T *>(p.out) + m * p.out_stride + n;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (p.bias != nullptr) sum[i] += static_cast<float>(reinterpret_cast<const T *>(p.bias)[n + i]);
    to[i] = E::narrow(sum[i]);
  }
}

template <class M, bool SPLIT>
void launch_linear_main(const LinearKP &kp, dim3 grid, hipStream_t stream) {
  if (kp.m <= 16)
    hipLaunchKernelGGL((linear_rows_kernel<M, 1, SPLIT>), grid, dim3(kLinearThreads), 0, stream, kp);
  else
    hipLaunchKernelGGL((linear_rows_kernel<M, 2, SPLIT>), grid, dim3(kLinearThreads), 0, stream, kp);
}

template <class M>
int launch_linear_typed(const LinearKP &kp, int splits, hipStream_t stream) {
  constexpr int TN = 16 * M::E::EPL;
  const dim3 grid((kp.n + TN - 1) / TN, splits);
  if (splits == 1) {
    launch_linear_main<M, false>(kp, grid, stream);
  } else {
    launch_linear_main<M, true>(kp, grid, stream);
    hipLaunchKernelGGL((linear_rows_sum_kernel<typename M::E>),
                       dim3((kp.n / 4 + kLinearSumThreads - 1) / kLinearSumThreads, kp.m), dim3(kLinearSumThreads), 0,
                       stream, kp, splits);
  }
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

int lane_block(int dtype) { return dtype == IC_DTYPE_F32 ? 4 : 8; }

}  // namespace

// k steps of a split, for `want` splits.  The rule (want == 0): a workgroup to a CU, at most 16 splits (their sums
// are read again), and none where each wave has four steps or fewer (the second launch costs more than they take).
// us with 1 / 2 / 4 / 8 / 16 splits, bf16, 16 rows: 4 096 x 4 096 28.4 / 20.0 / 14.9 / 12.2 / 14.5, 4 096 x 8 192
// 29.4 / 20.9 / 18.5 / 19.0 / 24.2, 11 008 x 4 096 75.9 / 44.0 / 28.3 / 21.9 / 24.2, 4 096 x 22 016 37.8 / 44.9 /
// 40.8 / 45.0 / 54.8, 1 024 x 1 024 6.8 / 7.4 / 7.4; fp32, 4 rows: 3 072 x 768 22.8 / 16.1 / 11.7 / 9.0 / 7.6 (24: 9.4).
static int linear_per_split(int n, int k, int dtype, int want) {
  const int nb = lane_block(dtype), steps = k / (4 * nb), tiles = (n + 16 * nb - 1) / (16 * nb);
  const int most = (steps + kLinearWaves - 1) / kLinearWaves;
  if (want <= 0) {
    want = most <= 4 ? 1 : device_cu_count() / tiles;
    want = want > 16 ? 16 : want;
  }
  want = want < 1 ? 1 : want > most ? most : want;
  return (steps + want - 1) / want;
}

int linear_rows_splits(int n, int k, int dtype, int want) {
  const int steps = k / (4 * lane_block(dtype)), per = linear_per_split(n, k, dtype, want);
  return (steps + per - 1) / per;
}

int launch_linear_rows(const LinearArgs &a, hipStream_t stream) {
  LinearKP kp;
  kp.x = (const char *)a.x;
  kp.w = (const char *)a.w;
  kp.bias = (const char *)a.bias;
  kp.out = (char *)a.out;
  kp.partials = (float *)a.workspace;
  kp.x_stride = a.x_stride;
  kp.w_stride = a.w_stride;
  kp.out_stride = a.out_stride;
  kp.m = a.m;
  kp.n = a.n;
  kp.steps = a.k / (4 * lane_block(a.dtype));
  kp.per_split = linear_per_split(a.n, a.k, a.dtype, a.splits);
  const int splits = (kp.steps + kp.per_split - 1) / kp.per_split;
  switch (a.dtype) {
    case IC_DTYPE_BF16: return launch_linear_typed<LinearBf16>(kp, splits, stream);
    case IC_DTYPE_F16: return launch_linear_typed<LinearF16>(kp, splits, stream);
    case IC_DTYPE_F32: return launch_linear_typed<LinearF32>(kp, splits, stream);
    default: return IC_ERR_UNSUPPORTED;
  }
}

}  // namespace ic
