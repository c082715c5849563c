// The two ends of a greedy decode step (examples/generate_text.py:27-40): the next token of each row from its
// logits, with the distance to the second best, and the bookkeeping of the step that follows it.
//
// Both are bound by launches and round trips, not by bytes (4 rows of 50 304 logits are 0.8 MB): torch's top-2, argmax
// and scatters are some thirty launches a token.  Here the rows are cut into chunks of kChunk logits, a workgroup
// each (52 workgroups for those 4 rows), and a second launch merges a row's chunks in one wave and stores the token; the
// bookkeeping (position, slot, context length, output column) is one launch.  GPT-2 small, fp32, batch 4, 128 + 64
// tokens with margins by graph replay: 45.3 -> 36.7 ms.
#include "ic_device.h"
#include "ic_internal.h"

namespace ic {

namespace {

constexpr int kChooseThreads = 256;
constexpr int kChunk = 4096;
constexpr int kMergeWaves = 16;

// The best of some logits, where it lies, and the second best.  NaN is the greatest (as for torch's argmax and topk);
// of equal logits the first one is the best, and the others are the second best.
struct Best {
  float v;
  int at;
  float second;
};

__device__ __forceinline__ bool above(float a, float b) { return a > b || (a != a && b == b); }
__device__ __forceinline__ float greater(float a, float b) { return above(b, a) ? b : a; }

__device__ __forceinline__ Best merge(const Best &a, const Best &b) {
  const bool other = above(b.v, a.v) || (!above(a.v, b.v) && b.at < a.at);
  return other ? Best{b.v, b.at, greater(a.v, b.second)} : Best{a.v, a.at, greater(a.second, b.v)};
}

__device__ __forceinline__ Best wave_best(Best x) {
#pragma unroll
  for (int step = 1; step < kWave; step *= 2) {
    const Best y{__shfl_xor(x.v, step, kWave), __shfl_xor(x.at, step, kWave), __shfl_xor(x.second, step, kWave)};
    x = merge(x, y);
  }
  return x;
}

// Below every logit: a logit of minus infinity is still the best of a row that has no other.
__device__ __forceinline__ Best none() { return {-__builtin_inff(), 0x7fffffff, -__builtin_inff()}; }

template <class E>
__global__ __launch_bounds__(kChooseThreads) void best_of_chunk_kernel(const char *logits, int64_t stride_bytes, int n,
                                                                       Best *bests) {
  constexpr int EPL = E::EPL;
  __shared__ Best s_best[kChooseThreads / kWave];
  const char *row = logits + blockIdx.y * stride_bytes;
  const int first = blockIdx.x * kChunk;
  Best best = none();
#pragma unroll
  for (int i = 0; i < kChunk / EPL / kChooseThreads; ++i) {
    const int at = first + (i * kChooseThreads + threadIdx.x) * EPL;
    if (at >= n) continue;  // (n is a multiple of EPL)
    float f[EPL];
    E::widen(load16(row + (int64_t)at * (16 / EPL)), f);
#pragma unroll
    for (int e = 0; e < EPL; ++e) best = merge(best, {f[e], at + e, -__builtin_inff()});
  }
  best = wave_best(best);
  if ((threadIdx.x & (kWave - 1)) == 0) s_best[threadIdx.x / kWave] = best;
  __syncthreads();
  if (threadIdx.x != 0) return;
#pragma unroll
  for (int w = 1; w < kChooseThreads / kWave; ++w) best = merge(best, s_best[w]);
  bests[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = best;
}

// A wave to a row.
__global__ __launch_bounds__(kMergeWaves *kWave) void choose_token_kernel(const ic_greedy_call p, const Best *bests,
                                                                          int chunks) {
  const int row = blockIdx.x * kMergeWaves + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if (row >= p.rows) return;
  const int64_t column = p.column != nullptr ? *p.column : 0;
  Best best = none();
  for (int c = lane; c < chunks; c += kWave) best = merge(best, bests[(int64_t)row * chunks + c]);
  best = wave_best(best);
  if (lane != 0) return;
  int64_t token = best.at;
  if (p.finished != nullptr) {
    if (p.finished[row]) token = p.eos;
    if (token == p.eos) p.finished[row] = 1;
  }
  if (p.next != nullptr) p.next[row] = token;
  if (column < 0 || column >= p.columns) return;
  if (p.tokens != nullptr) p.tokens[row * p.token_stride + column] = token;
  if (p.margins != nullptr) p.margins[row * p.margin_stride + column] = best.v - best.second;
}

__global__ __launch_bounds__(kChooseThreads) void advance_rows_kernel(const ic_advance_call p) {
  const int row = blockIdx.x * kChooseThreads + threadIdx.x;
  if (row == 0 && p.column != nullptr) *p.column += 1;
  if (row >= p.rows) return;
  const int position = p.context_lens[row];
  p.context_lens[row] = position + 1;
  p.positions[row] = position;
  p.token_positions[row] = position;
  const int block = position / p.block_size;
  p.slot_mapping[row] = position < 0 || block >= p.table_width
                            ? -1
                            : (int64_t)p.block_tables[row * p.block_table_stride + block] * p.block_size +
                                  position % p.block_size;
}

int chunks_of(int n) { return (n + kChunk - 1) / kChunk; }

template <class E>
void launch_bests(const ic_greedy_call &a, Best *bests, hipStream_t stream) {
  constexpr int kMostRows = 65535;  // gridDim.y
  for (int row = 0; row < a.rows; row += kMostRows) {
    const int rows = a.rows - row < kMostRows ? a.rows - row : kMostRows;
    const int64_t stride = a.stride * (16 / E::EPL);
    hipLaunchKernelGGL(best_of_chunk_kernel<E>, dim3(chunks_of(a.n), rows), dim3(kChooseThreads), 0, stream,
                       (const char *)a.logits + row * stride, stride, a.n, bests + (int64_t)row * chunks_of(a.n));
  }
}

}  // namespace

size_t greedy_workspace_bytes(int rows, int n) { return (size_t)rows * chunks_of(n) * sizeof(Best); }

int launch_greedy(const ic_greedy_call &a, hipStream_t stream) {
  Best *bests = static_cast<Best *>(a.workspace);
  switch (a.dtype) {
    case IC_DTYPE_BF16: launch_bests<Bf16>(a, bests, stream); break;
    case IC_DTYPE_F16: launch_bests<F16>(a, bests, stream); break;
    case IC_DTYPE_F32: launch_bests<F32>(a, bests, stream); break;
    default: return IC_ERR_UNSUPPORTED;
  }
  hipLaunchKernelGGL(choose_token_kernel, dim3((a.rows + kMergeWaves - 1) / kMergeWaves), dim3(kMergeWaves * kWave), 0,
                     stream, a, bests, chunks_of(a.n));
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

int launch_advance(const ic_advance_call &a, hipStream_t stream) {
  hipLaunchKernelGGL(advance_rows_kernel, dim3((a.rows + kChooseThreads - 1) / kChooseThreads), dim3(kChooseThreads), 0,
                     stream, a);
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

}  // namespace ic
