// The linears of a decode step with what stands around them in a transformer layer
// (ironcore/models/transformer.py:77-135), for up to 32 rows:
//   out = act(x W + bias)                                    up-projection, output layer
//   [q | k | v] = x W + bias, rotated, k and v stored into the pool
//   out = x W + bias + residual, norm_out = norm(out)        attention output, down-projection
//
// Bound by the stream over W and, for small models, by the 2-4 us between two dependent launches
// (drain, start, a cold round trip to the weights): activation, append, residual and norm ride on
// the launches that the product has anyway.
//
//  * MFMA with W as the A operand, x as B (as in linear_rows.hip): a lane loads KR rows x NB columns of W, 16
//    lanes side by side.  NB sets the width of a workgroup's tile (16 * NB columns).
//  * 8 waves take the k steps in turn, D of them in flight, and add up through LDS.
//  * A CU has some 250 cache lines on their way at most (measured: 12 to 256 workgroups read at 30-36 bytes/ns each by
//    whole lines, 15 by half lines), so the weights of a large model need all CUs and rows of 256 bytes, those of a small
//    one as few launches as possible.  Columns that fill the CUs are done in one launch; else k is split over
//    workgroups and a second launch adds the partial sums (fp32) in a fixed order, with everything that follows.
//    A norm needs whole rows, so its launch has a workgroup to a row, and the product before it is always split.
//
// A layer with plain attention is 7-10 launches instead of 17-19: 2 for each product with a norm, 1 or 2 (split) for the
// projections and the up-projection, 1 or 2 for attention.  GPT-2 small, fp32, batch 4, 128 + 64 tokens by graph replay 66.5 -> 45.3 ms;
// a Llama-dims step (four layers, batch 16, bf16) 866 -> 768 us; one of 2 layers, d_model 2 048, 321 -> 140.
#include "ic_device.h"
#include "ic_internal.h"
#include "rope_device.h"
#include "step_common.h"
#include "../../include/ironcore_paged.h"

namespace ic {

using namespace step;

namespace {

struct StepKP {
  const char *x, *norm_weight, *norm_bias, *residual;
  const char *w[2], *bias[2];
  char *out, *norm_out;
  float *partials;     // [splits][m][n[0] + n[1]]
  int64_t x_stride, out_stride, norm_out_stride, residual_stride, w_stride[2];  // elements
  int n[2];            // columns of the two matrices (n[1] = 0: one)
  int m, tiles, tiles0;  // tiles0: tiles of the first matrix
  int steps, per_split, splits;  // k in steps
  int norm, act, gated;
  float eps;
  // the append: columns [0, hn * hd) are queries, gn * hd keys and gn * hd values follow
  char *k_pool, *v_pool;
  const int64_t *slots;
  const int32_t *positions;
  const float *cos_table, *sin_table;
  int64_t sb, sh, st, num_slots, table_rows;  // pool strides in elements
  int hn, gn, hd, block_size;
};

// What the end of a product needs beside its sums, fetched before them: the bias of two neighbouring columns (and of
// their gates), and where a row's new keys and values go.
struct Extras {
  float a = 0.f, b = 0.f, gate_a = 0.f, gate_b = 0.f;
};
struct Place {
  int64_t slot = -1, angle = 0;  // pool slot; first element of the row's rotary tables
};

template <class E>
__device__ __forceinline__ Extras fetch_extras(const StepKP &p, int col) {
  Extras x;
  const int mat = col >= p.n[0] ? 1 : 0;
  const typename E::type *bias = reinterpret_cast<const typename E::type *>(p.bias[mat]);
  if (bias == nullptr) return x;
  bias += col - (mat ? p.n[0] : 0);
  x.a = static_cast<float>(bias[0]), x.b = static_cast<float>(bias[1]);
  if (p.gated) x.gate_a = static_cast<float>(bias[p.n[0] / 2]), x.gate_b = static_cast<float>(bias[p.n[0] / 2 + 1]);
  return x;
}

__device__ __forceinline__ Place fetch_place(const StepKP &p, int row) {
  Place at;
  if (p.slots == nullptr) return at;
  at.slot = p.slots[row];
  if (p.cos_table == nullptr) return at;
  const int64_t pos = p.positions[row];
  at.angle = (pos < 0 ? 0 : pos >= p.table_rows ? p.table_rows - 1 : pos) * (p.hd / 2);
  return at;
}

// Two neighbouring columns of the projections [q | k | v] of row `row`, rotated and stored where they belong.
template <class E>
__device__ __forceinline__ void store_qkv(const StepKP &p, int row, int col, float a, float b, const Place &place) {
  using T = typename E::type;
  const int q_cols = p.hn * p.hd, kv_cols = p.gn * p.hd;
  const bool value = col >= q_cols + kv_cols;
  if (p.cos_table != nullptr && !value) {
    const int64_t at = place.angle + (col % p.hd) / 2;
    rotate_pair(a, b, p.cos_table[at], p.sin_table[at], a, b);
  }
  const Pair<T> v{E::narrow(a), E::narrow(b)};
  if (col < q_cols) {
    *reinterpret_cast<Pair<T> *>(reinterpret_cast<T *>(p.out) + row * p.out_stride + col) = v;
    return;
  }
  const int64_t slot = place.slot;
  if (slot < 0 || slot >= p.num_slots) return;
  const int64_t blk = (p.num_slots >> 32) != 0 ? slot / p.block_size : (uint32_t)slot / (uint32_t)p.block_size;
  const int at = col - q_cols - (value ? kv_cols : 0);
  T *pool = reinterpret_cast<T *>(value ? p.v_pool : p.k_pool);
  *reinterpret_cast<Pair<T> *>(pool + blk * p.sb + (at / p.hd) * p.sh + (slot - blk * p.block_size) * p.st + at % p.hd) = v;
}

// Two neighbouring columns of a row, their sums complete but for the bias: bias, activation (with the gate that
// belongs to a feature), rotation, and the store.  `col` counts over both matrices, or over the features.
template <class E>
__device__ __forceinline__ void finish_pair(const StepKP &p, int row, int col, float a, float b, float ga, float gb,
                                            const Extras &x, const Place &place) {
  using T = typename E::type;
  a += x.a, b += x.b;
  if (p.gated) {
    ga += x.gate_a, gb += x.gate_b;
    if (p.act == IC_ACT_SWIGLU) {
      a = a * sigmoid(a) * ga, b = b * sigmoid(b) * gb;
    } else {
      a *= sigmoid(ga), b *= sigmoid(gb);
    }
  } else if (p.act != IC_ACT_NONE) {
    a = activate(p.act, a), b = activate(p.act, b);
  }
  if (p.slots != nullptr)
    store_qkv<E>(p, row, col, a, b, place);
  else
    *reinterpret_cast<Pair<T> *>(reinterpret_cast<T *>(p.out) + row * p.out_stride + col) =
        Pair<T>{E::narrow(a), E::narrow(b)};
}

template <class M, int MT, int NB, bool SPLIT>
__global__ __launch_bounds__(kStepThreads) void step_linear_kernel(const StepKP p) {
  using E = typename M::E;
  using S = Shape<M, NB>;
  constexpr int D = S::D, KR = S::KR, ES = S::ES, TN = S::TN, PITCH = S::PITCH;
  __shared__ __align__(16) float s_sum[kStepWaves * 16 * PITCH];
  // tile of the workgroup: workgroups go round the XCDs, neighbouring tiles to one of them
  const int per_xcd = (p.tiles + kXcds - 1) / kXcds;
  const int tile = (int)(blockIdx.x % kXcds) * per_xcd + (int)(blockIdx.x / kXcds);
  if (tile >= p.tiles) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int c = lane & 15, g = lane >> 4;
  const int mat = tile >= p.tiles0 ? 1 : 0;
  const int n = p.n[mat];
  // columns of the tile: with a gated activation TN / 2 features, then the TN / 2 gates that belong to them
  const bool gated = !SPLIT && p.gated;
  const int half = n / 2;
  const int n0 = (tile - (mat ? p.tiles0 : 0)) * (gated ? TN / 2 : TN);
  int col;  // (columns past the end: loaded, never stored)
  if (gated) {
    col = n0 + (c & 7) * NB;
    col = (col < half ? col : half - NB) + (c >> 3) * half;
  } else {
    col = n0 + c * NB < n ? n0 + c * NB : n - NB;
  }
  const int64_t w_stride = p.w_stride[mat];
  const char *w = p.w[mat] + ((int64_t)g * KR * w_stride + col) * ES;
  const int first = SPLIT ? blockIdx.y * p.per_split + wave : wave;
  const int end_step = SPLIT ? ((int)(blockIdx.y + 1) * p.per_split < p.steps ? (int)(blockIdx.y + 1) * p.per_split : p.steps)
                             : p.steps;
  const int mine = first < end_step ? (end_step - first + kStepWaves - 1) / kStepWaves : 0;  // steps of this wave
  Words<S::NW> wv[D][KR];
  Vec16 xv[D][MT];
  const char *x[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int row = t * 16 + c < p.m ? t * 16 + c : p.m - 1;
    x[t] = p.x + (row * p.x_stride + g * KR) * ES;
  }
  auto load = [&](int i, int d) {
    const int step = first + i * kStepWaves;
    const char *at = w + (int64_t)step * S::STEP * w_stride * ES;
#pragma unroll
    for (int r = 0; r < KR; ++r) wv[d][r] = *reinterpret_cast<const Words<S::NW> *>(at + r * w_stride * ES);
#pragma unroll
    for (int t = 0; t < MT; ++t) xv[d][t] = load16(x[t] + (int64_t)step * 64);
  };
  // The sums' end: a thread takes the same two columns of every row it has (widths are powers of two).
  const int cols = gated ? TN / 2 : TN, end = gated ? half : n;
  const int before = mat ? p.n[0] : 0;
  const int at = 2 * (threadIdx.x % (cols / 2)), first_row = threadIdx.x / (cols / 2), row_step = kStepThreads / (cols / 2);
  Extras extras;
  Place place;
  if constexpr (!SPLIT) {  // (on their way with the first steps)
    if (n0 + at < end) extras = fetch_extras<E>(p, before + n0 + at);
    if (first_row < p.m) place = fetch_place(p, first_row);
  }
  f32x4_t acc[NB][MT];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[j][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto add = [&](int d) { multiply<M, MT, NB>(wv[d], xv[d], acc); };
  if (mine >= D) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, d);
    int i = D;
    for (; i + D <= mine; i += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        add(d);
        load(i + d, d);
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      add(d);
      if (i + d < mine) load(i + d, d);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (i + d < mine) add(d);
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d < mine) load(d, d);
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d < mine) add(d);
  }
  // ---- the waves' sums, 16 rows of x at a time, two columns a thread --------------------------
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (t > 0) __syncthreads();
    float *to = s_sum + (wave * 16 + c) * PITCH + g * 4 * NB;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NB; ++j) to[r * NB + j] = acc[j][t][r];
    __syncthreads();
    for (int r = first_row; r < 16; r += row_step) {
      const int row = t * 16 + r;
      if (row >= p.m || n0 + at >= end) continue;
      auto total = [&](int column, float &a, float &b) {
        a = b = 0.f;
#pragma unroll
        for (int v = 0; v < kStepWaves; ++v) {
          const float2 s = *reinterpret_cast<const float2 *>(s_sum + (v * 16 + r) * PITCH + column);
          a += s.x, b += s.y;
        }
      };
      float a, b, ga = 0.f, gb = 0.f;
      total(at, a, b);
      if constexpr (SPLIT) {
        *reinterpret_cast<float2 *>(p.partials + ((int64_t)blockIdx.y * p.m + row) * (p.n[0] + p.n[1]) + before + n0 +
                                    at) = make_float2(a, b);
      } else {
        if (gated) total(TN / 2 + at, ga, gb);
        finish_pair<E>(p, row, before + n0 + at, a, b, ga, gb, extras, row == first_row ? place : fetch_place(p, row));
      }
    }
  }
}

// ---- the second launch of a split product ------------------------------------------------------

// The splits' partial sums in order, eight on their way at a time (a split past the last: loaded again, not added).
__device__ __forceinline__ float4 sum_partials(const float *at, int64_t pitch, int splits) {
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s = 0; s < splits; s += 8) {
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = *reinterpret_cast<const float4 *>(at + (s + i < splits ? s + i : splits - 1) * pitch);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (s + i < splits) sum.x += v[i].x, sum.y += v[i].y, sum.z += v[i].z, sum.w += v[i].w;
    }
  }
  return sum;
}

constexpr int kFinishThreads = 128;

// Four columns a lane.  Bound by the round trips.
template <class E>
__global__ __launch_bounds__(kFinishThreads) void step_finish_kernel(const StepKP p) {
  const int col = (blockIdx.x * kFinishThreads + threadIdx.x) * 4, row = blockIdx.y;
  const int total = p.n[0] + p.n[1], cols = p.gated ? total / 2 : total;
  if (col >= cols) return;
  const float *at = p.partials + (int64_t)row * total + col;
  const int64_t pitch = (int64_t)p.m * total;
  const Extras low = fetch_extras<E>(p, col), high = fetch_extras<E>(p, col + 2);
  const Place place = fetch_place(p, row);
  const float4 v = sum_partials(at, pitch, p.splits);
  float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
  if (p.gated) g = sum_partials(at + cols, pitch, p.splits);
  finish_pair<E>(p, row, col, v.x, v.y, g.x, g.y, low, place);
  finish_pair<E>(p, row, col + 2, v.z, v.w, g.z, g.w, high, place);
}

constexpr int kRowThreads = 1024;

// Sum over the workgroup; every thread has the total.
__device__ __forceinline__ float block_sum(float x, float *s) {
  x = group_sum<kWave>(x);
  if (blockDim.x == kWave) return x;
  const int wave = threadIdx.x / kWave;
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) s[wave] = x;
  __syncthreads();
  float sum = 0.f;
  for (int i = 0; i < (int)blockDim.x / kWave; ++i) sum += s[i];
  return sum;
}

// A workgroup to a row: out = sums + bias + residual, rounded to the element type, and its norm.  ITER * 4 columns a
// thread stay in registers between the passes (mean, variance, output).  Bound by the round trips.
template <class E, int ITER>
__global__ __launch_bounds__(kRowThreads) void step_rows_kernel(const StepKP p) {
  using T = typename E::type;
  struct alignas(4 * sizeof(T)) Quad {
    T e[4];
  };
  __shared__ float s_red[kRowThreads / kWave];
  const int n = p.n[0], row = blockIdx.x;
  float v[ITER][4];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < ITER; ++i) {
    const int col = (i * blockDim.x + threadIdx.x) * 4;
    const bool in = col < n;
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
    Quad bias{}, res{};
    if (in) {
      if (p.bias[0] != nullptr) {
        const T *from = reinterpret_cast<const T *>(p.bias[0]) + col;
#pragma unroll
        for (int e = 0; e < 4; ++e) bias.e[e] = from[e];
      }
      if (p.residual != nullptr)
        res = *reinterpret_cast<const Quad *>(reinterpret_cast<const T *>(p.residual) + row * p.residual_stride + col);
      t = sum_partials(p.partials + (int64_t)row * n + col, (int64_t)p.m * n, p.splits);
    }
    const float f[4] = {t.x, t.y, t.z, t.w};
    Quad h;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h.e[e] = E::narrow(f[e] + static_cast<float>(bias.e[e]) + static_cast<float>(res.e[e]));
      v[i][e] = in ? static_cast<float>(h.e[e]) : 0.f;
      sum += v[i][e];
    }
    if (in && p.out != nullptr) *reinterpret_cast<Quad *>(reinterpret_cast<T *>(p.out) + row * p.out_stride + col) = h;
  }
  if (p.norm == IC_NORM_NONE) return;
  Quad gain[ITER], shift[ITER];  // on their way while the sums are taken
#pragma unroll
  for (int i = 0; i < ITER; ++i) {
    const int col = (i * blockDim.x + threadIdx.x) * 4;
    shift[i] = Quad{};
    if (col < n) {
      gain[i] = *reinterpret_cast<const Quad *>(reinterpret_cast<const T *>(p.norm_weight) + col);
      if (p.norm_bias != nullptr) shift[i] = *reinterpret_cast<const Quad *>(reinterpret_cast<const T *>(p.norm_bias) + col);
    }
  }
  const float inv_n = 1.f / (float)n;
  const float mean = p.norm == IC_NORM_LAYER ? block_sum(sum, s_red) * inv_n : 0.f;
  float squares = 0.f;
#pragma unroll
  for (int i = 0; i < ITER; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if ((int)(i * blockDim.x + threadIdx.x) * 4 < n)
        squares = __builtin_fmaf(v[i][e] - mean, v[i][e] - mean, squares);
  const float scale = 1.f / sqrtf(block_sum(squares, s_red) * inv_n + p.eps);
#pragma unroll
  for (int i = 0; i < ITER; ++i) {
    const int col = (i * blockDim.x + threadIdx.x) * 4;
    if (col >= n) continue;
    Quad y;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      y.e[e] = E::narrow((v[i][e] - mean) * scale * static_cast<float>(gain[i].e[e]) + static_cast<float>(shift[i].e[e]));
    *reinterpret_cast<Quad *>(reinterpret_cast<T *>(p.norm_out) + row * p.norm_out_stride + col) = y;
  }
}

template <class E>
void launch_rows(const StepKP &kp, hipStream_t stream) {
  const int quads = (kp.n[0] + 3) / 4;
  const int threads = quads >= kRowThreads ? kRowThreads : (quads + kWave - 1) / kWave * kWave;
  switch ((quads + threads - 1) / threads) {
    case 1: hipLaunchKernelGGL((step_rows_kernel<E, 1>), dim3(kp.m), dim3(threads), 0, stream, kp); break;
    case 2: hipLaunchKernelGGL((step_rows_kernel<E, 2>), dim3(kp.m), dim3(threads), 0, stream, kp); break;
    default: hipLaunchKernelGGL((step_rows_kernel<E, 4>), dim3(kp.m), dim3(threads), 0, stream, kp); break;
  }
}

template <class M, int MT, int NB>
void launch_product(const StepKP &kp, hipStream_t stream) {
  const dim3 grid((kp.tiles + kXcds - 1) / kXcds * kXcds, kp.partials ? kp.splits : 1);
  if (kp.partials != nullptr)
    hipLaunchKernelGGL((step_linear_kernel<M, MT, NB, true>), grid, dim3(kStepThreads), 0, stream, kp);
  else
    hipLaunchKernelGGL((step_linear_kernel<M, MT, NB, false>), grid, dim3(kStepThreads), 0, stream, kp);
}

template <class M>
int launch_typed(StepKP &kp, int tile_bytes, bool rows, hipStream_t stream) {
  constexpr int W = sizeof(typename M::E::type) == 2 ? 2 : 1;  // NB of 64 bytes
  if (kp.w[0] != nullptr) {
    const bool one = kp.m <= 16;
    switch (tile_bytes) {
      case 64: one ? launch_product<M, 1, W>(kp, stream) : launch_product<M, 2, W>(kp, stream); break;
      case 128: one ? launch_product<M, 1, 2 * W>(kp, stream) : launch_product<M, 2, 2 * W>(kp, stream); break;
      default: one ? launch_product<M, 1, 4 * W>(kp, stream) : launch_product<M, 2, 4 * W>(kp, stream); break;
    }
  }
  if (rows) {
    launch_rows<typename M::E>(kp, stream);
  } else if (kp.partials != nullptr) {
    const int cols = kp.gated ? kp.n[0] / 2 : kp.n[0] + kp.n[1];
    hipLaunchKernelGGL((step_finish_kernel<typename M::E>),
                       dim3((cols / 4 + kFinishThreads - 1) / kFinishThreads, kp.m), dim3(kFinishThreads), 0, stream, kp);
  }
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

}  // namespace

StepPlan step_linear_plan(const ic_step_linear_call &a) {
  StepPlan plan;
  const bool rows = a.residual != nullptr || a.norm != IC_NORM_NONE;
  const int es = elem_size(a.dtype), steps = a.k * es / 64;
  const bool gated = a.act >= IC_ACT_GLU;
  // The rule, from both sides in us (tile bytes / splits, both launches, W from memory):
  //  * whole rows follow: 8 splits (one batch of loads in the second launch) or as many as the CUs hold, tiles of 128
  //    bytes while 32 of them hold a row.  fp32, 4 rows: 768 x 768 64/8 6.5, 128/8 6.6, 256/8 6.8, 128/1 9.1, 128/16 8.3;
  //    3 072 x 768 128/8 8.8, 64/8 9.1, 256/16 9.3; bf16, 16 rows: 4 096 x 4 096 256/8 15.0, 128/4 15.4, 64/2 17.3,
  //    11 008 x 4 096 256/8 23.9, 128/4 25.4; 32 rows 2 048 x 2 048 128/8 9.8, 256/8 10.4.
  //  * short columns: one launch of narrow tiles, since a launch more costs what it saves.  fp32, 4 rows 768 x 2 304 64/1
  //    6.4, 128/1 7.5, 256/6 8.0, 768 x 3 072 64/1 6.7, 256/4 9.2; bf16, 4 rows 1 024 x 3 072 64/1 6.9, 256/8 7.7, 1 024 x
  //    5 504 gated 64/1 8.0, 128/1 8.9, 256/1 9.6.
  //  * long ones: whole lines and all CUs.  bf16, 32 rows 2 048 x 6 144 256/5 13.6, 64/1 14.8, 2 048 x 11 008 gated 256/2
  //    17.7, 128/1 19.2; 16 rows 4 096 x 12 288 256/2 24.7, 128/1 26.4, 4 096 x 22 016 gated 256/1 39.3, 128/2 44.6.
  const int64_t row_bytes = (int64_t)(a.n + a.n2) * es;
  const bool narrow = !rows && a.k <= 1536 && row_bytes <= 64 * 2 * (int64_t)device_cu_count();
  plan.tile_bytes = a.tile_bytes > 0 ? a.tile_bytes : narrow ? 64 : rows && row_bytes <= 32 * 128 ? 128 : 256;
  const int cols = plan.tile_bytes / es;
  const int most = (steps + kStepWaves - 1) / kStepWaves;  // splits with a step for every wave
  plan.splits = a.splits;
  if (a.splits <= 0) {
    plan.splits = narrow ? 1 : device_cu_count() / ((a.n + a.n2 + cols - 1) / cols);
    plan.splits = plan.splits > 8 ? 8 : plan.splits > most ? most : plan.splits;
    if (plan.splits < 1) plan.splits = 1;
  }
  plan.rows = rows;
  if (a.w == nullptr) {  // the norm alone
    plan.partial = false, plan.splits = plan.per_split = plan.tiles = plan.tiles0 = 0;
    return plan;
  }
  plan.per_split = (steps + plan.splits - 1) / plan.splits;
  plan.splits = (steps + plan.per_split - 1) / plan.per_split;
  plan.partial = rows || plan.splits > 1;
  const int own = gated && !plan.partial ? cols / 2 : cols, n = gated && !plan.partial ? a.n / 2 : a.n;
  plan.tiles0 = (n + own - 1) / own;
  plan.tiles = plan.tiles0 + (a.n2 + own - 1) / own;
  return plan;
}

int launch_step_linear(const ic_step_linear_call &a, hipStream_t stream) {
  const StepPlan plan = step_linear_plan(a);
  StepKP kp;
  kp.x = (const char *)a.x, kp.norm_weight = (const char *)a.norm_weight, kp.norm_bias = (const char *)a.norm_bias;
  kp.residual = (const char *)a.residual;
  kp.w[0] = (const char *)a.w, kp.w[1] = (const char *)a.w2;
  kp.bias[0] = a.w ? (const char *)a.bias : nullptr, kp.bias[1] = (const char *)a.bias2;
  kp.w_stride[0] = a.w_stride, kp.w_stride[1] = a.w2_stride;
  kp.n[0] = a.n, kp.n[1] = a.n2;
  kp.out = (char *)a.out, kp.norm_out = (char *)a.norm_out;
  kp.partials = plan.partial ? (float *)a.workspace : nullptr;
  kp.x_stride = a.x_stride, kp.out_stride = a.out_stride, kp.residual_stride = a.residual_stride;
  kp.norm_out_stride = a.norm_out_stride;
  kp.m = a.m, kp.tiles = plan.tiles, kp.tiles0 = plan.tiles0;
  kp.steps = a.k * elem_size(a.dtype) / 64, kp.per_split = plan.per_split, kp.splits = plan.splits;
  kp.norm = a.norm, kp.act = a.act, kp.gated = a.act >= IC_ACT_GLU, kp.eps = a.eps;
  kp.k_pool = (char *)a.k_pool, kp.v_pool = (char *)a.v_pool;
  kp.slots = a.slot_mapping, kp.positions = a.positions;
  kp.cos_table = a.cos_table, kp.sin_table = a.sin_table, kp.table_rows = a.table_rows;
  kp.sb = a.pool_stride_block, kp.sh = a.pool_stride_head, kp.st = a.pool_stride_token;
  kp.num_slots = a.num_blocks * a.block_size;
  kp.hn = a.hn, kp.gn = a.gn, kp.hd = a.hd, kp.block_size = a.block_size;
  switch (a.dtype) {
    case IC_DTYPE_BF16: return launch_typed<StepBf16>(kp, plan.tile_bytes, plan.rows, stream);
    case IC_DTYPE_F16: return launch_typed<StepF16>(kp, plan.tile_bytes, plan.rows, stream);
    case IC_DTYPE_F32: return launch_typed<StepF32>(kp, plan.tile_bytes, plan.rows, stream);
    default: return IC_ERR_UNSUPPORTED;
  }
}

}  // namespace ic
