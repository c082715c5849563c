// Rotary position embedding fused into the KV append.
//
// A transformer layer with rotary embeddings rotates its query and key rows
// right after the projections and before attention
// (reference: ironcore/models/transformer.py:95-98 calling
// ironcore/layers/positional_embedding/rotary.py:53-83).  With a block KV
// cache that is also the moment the new K/V rows enter the pool, so one pass
// does all three: rotate Q in place, rotate K into its pool slots, copy V into
// its pool slots.  Rotated keys are stored, so a cached key is never rotated
// again.
//
// Arithmetic is the reference's (rotary.py:69-83), element pairs (2i, 2i+1):
//     out[2i]   = x[2i] * cos - x[2i+1] * sin
//     out[2i+1] = x[2i] * sin + x[2i+1] * cos
// in fp32 with every product and sum rounded on its own (no fused
// multiply-add), then rounded to the element type: bit-identical to the same
// expression evaluated by torch on the CPU.  cos/sin come from the caller's
// fp32 tables [rows, hd/2] (the reference caches exactly such tables,
// rotary.py:36-51), indexed by positions[token]: WHICH row a token uses is the
// caller's decision (its true position in the sequence for a cached decoder).
//
// HBM-bound: one lane handles one 16-byte chunk (4 pairs in 16-bit types, 2
// in fp32) and the matching 16 or 8 bytes of each table row; rows of few
// chunks share a workgroup; blockIdx.z picks K, V or Q.  Algorithmic traffic:
// K and V rows read once and written once, Q rows read and written in place,
// 12 bytes of slot and position per token; the table rows in use stay in cache.
#include "append_rows.h"
#include "ic_internal.h"
#include "rope_device.h"
#include "../../include/ironcore_paged.h"

namespace ic {

namespace {

struct RopeKP {
  const char *q;          // or nullptr
  char *q_out;            // where its rotated rows go (q itself: in place)
  const char *k_new;      // or nullptr: no K/V work
  const char *v_new;
  char *k_pool;
  char *v_pool;
  const int64_t *slot_mapping;
  const int32_t *positions;
  const float *cos_table;
  const float *sin_table;
  int64_t q_stride_bytes;
  int64_t q_out_stride_bytes;
  int64_t new_stride_bytes;
  int64_t stride_block_bytes;
  int64_t stride_head_bytes;
  int64_t stride_token_bytes;
  int64_t num_slots;
  int64_t table_rows;
  int chunks_per_head;
  int q_chunks;   // per token
  int kv_chunks;  // per token
  int q_row_shift;   // lanes of a row in a workgroup
  int kv_row_shift;
  int block_size;
  int half_hd;
};

template <class E, bool WIDE>
__global__ __launch_bounds__(kAppendThreads) void rope_kv_append_kernel(const RopeKP p, int64_t t0, int64_t n_tokens,
                                                                             const ZeroRows zero) {
  if (zero_part(zero, p.q_chunks > 0 ? 3 : 2)) return;
  constexpr int PAIRS = E::EPL / 2;  // pairs in one 16-byte chunk
  const int part = blockIdx.z;  // 0: K, 1: V, 2: Q
  const int row_shift = part == 2 ? p.q_row_shift : p.kv_row_shift;
  const int64_t t = t0 + append_token<WIDE>(row_shift);
  const int c = append_chunk<WIDE>(row_shift);
  if (t >= n_tokens) return;
  int64_t pos = p.positions[t];
  pos = pos < 0 ? 0 : pos;
  pos = pos >= p.table_rows ? p.table_rows - 1 : pos;
  if (part == 2) {
    if (p.q == nullptr || c >= p.q_chunks) return;
    const int within = c % p.chunks_per_head;
    const int64_t trig = pos * p.half_hd + within * PAIRS;
    store16(p.q_out + t * p.q_out_stride_bytes + (int64_t)c * 16,
            rotate_chunk<E>(load16(p.q + t * p.q_stride_bytes + (int64_t)c * 16), p.cos_table + trig, p.sin_table + trig));
    return;
  }
  if (p.k_new == nullptr || c >= p.kv_chunks) return;
  const int64_t slot = p.slot_mapping[t];
  if (slot < 0 || slot >= p.num_slots) return;
  const int64_t blk = slot_block<WIDE>(slot, p.block_size, p.num_slots);
  const int64_t off = slot - blk * p.block_size;
  const int head = c / p.chunks_per_head;
  const int within = c - head * p.chunks_per_head;
  const int64_t dst = blk * p.stride_block_bytes + head * p.stride_head_bytes + off * p.stride_token_bytes +
                      (int64_t)within * 16;
  const int64_t src = t * p.new_stride_bytes + (int64_t)c * 16;
  if (part == 1) {
    store16(p.v_pool + dst, load16(p.v_new + src));
  } else {
    const int64_t trig = pos * p.half_hd + within * PAIRS;
    store16(p.k_pool + dst, rotate_chunk<E>(load16(p.k_new + src), p.cos_table + trig, p.sin_table + trig));
  }
}

template <class E>
int launch_typed(const RopeKP &kp, int64_t n_tokens, ZeroRows zero, hipStream_t stream) {
  const int widest = kp.q_chunks > kp.kv_chunks ? kp.q_chunks : kp.kv_chunks;
  const int shift = kp.q_row_shift > kp.kv_row_shift ? kp.q_row_shift : kp.kv_row_shift;
  const int rows = kAppendThreads >> shift;  // token rows of a workgroup, at least
  dim3 grid((widest + kAppendThreads - 1) / kAppendThreads, 1, kp.q_chunks > 0 ? 3 : 2);
  const bool wide = kp.kv_row_shift == kAppendThreadsShift && (kp.q_chunks == 0 || kp.q_row_shift == kAppendThreadsShift);
  const int64_t slice = (int64_t)65535 * rows;  // gridDim.y limit: walk longer batches in slices
  const unsigned parts = grid.z;
  for (int64_t t0 = 0; t0 < n_tokens; t0 += slice) {
    const int64_t n = n_tokens - t0 < slice ? n_tokens - t0 : slice;
    grid.y = (unsigned)((n + rows - 1) / rows);
    grid.z = parts + zero_slices(zero, grid);
    hipLaunchKernelGGL((wide ? rope_kv_append_kernel<E, true> : rope_kv_append_kernel<E, false>), grid, dim3(kAppendThreads), 0, stream, kp, t0, t0 + n, zero);
    zero.total = 0;  // the first slice's
  }
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

}  // namespace

int launch_rope_kv_append(const RopeAppendArgs &a, hipStream_t stream) {
  if (a.append.n_tokens == 0) return IC_OK;
  const AppendArgs &ap = a.append;
  const int es = elem_size(ap.dtype);
  RopeKP kp;
  kp.q = (const char *)a.q;
  kp.q_out = (char *)a.q_out;
  kp.k_new = (const char *)ap.k_new;
  kp.v_new = (const char *)ap.v_new;
  kp.k_pool = (char *)ap.k_pool;
  kp.v_pool = (char *)ap.v_pool;
  kp.slot_mapping = ap.slot_mapping;
  kp.positions = a.positions;
  kp.cos_table = a.cos_table;
  kp.sin_table = a.sin_table;
  kp.q_stride_bytes = a.q_stride_token * es;
  kp.q_out_stride_bytes = a.q_out_stride_token * es;
  kp.new_stride_bytes = ap.new_stride_token * es;
  kp.stride_block_bytes = ap.pool.stride_block * es;
  kp.stride_head_bytes = ap.pool.stride_head * es;
  kp.stride_token_bytes = ap.pool.stride_token * es;
  kp.num_slots = ap.pool.num_blocks * ap.pool.block_size;
  kp.table_rows = a.table_rows;
  kp.chunks_per_head = ap.hd * es / 16;
  kp.q_chunks = a.q ? kp.chunks_per_head * a.hn : 0;
  kp.kv_chunks = ap.k_new ? kp.chunks_per_head * ap.gn : 0;
  kp.q_row_shift = append_row_shift(kp.q_chunks);
  kp.kv_row_shift = append_row_shift(kp.kv_chunks);
  kp.block_size = ap.pool.block_size;
  kp.half_hd = ap.hd / 2;
  switch (ap.dtype) {
    case IC_DTYPE_BF16: return launch_typed<Bf16>(kp, ap.n_tokens, ap.zero, stream);
    case IC_DTYPE_F16: return launch_typed<F16>(kp, ap.n_tokens, ap.zero, stream);
    case IC_DTYPE_F32: return launch_typed<F32>(kp, ap.n_tokens, ap.zero, stream);
    default: return IC_ERR_UNSUPPORTED;
  }
}

}  // namespace ic
