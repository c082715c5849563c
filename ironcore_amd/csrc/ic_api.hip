// C ABI: argument validation on the host, then dispatch to the kernel
// launchers.  Nothing here synchronises or keeps state, and nothing but
// ic_step_status allocates.
#include <atomic>
#include <cstring>

#include "ic_internal.h"
#include "../../include/ironcore_paged.h"

namespace ic {
namespace decode {
long long decode_occupancy_queries();  // paged_decode_mfma.hip
}
}  // namespace ic

// Device memory of the entry point that may not allocate (ic_paged_decode_static): the decode
// workspace (row prefix sums and split-K partials) lives in this array instead of a buffer the
// caller brings.  Every GPU the library runs on holds its own copy at its own address until the
// process ends; host code reaches it only through the address hipGetSymbolAddress returns for the
// current device (static_scratch below), never through the array's name.
static __device__ __align__(256) unsigned char scratch[IC_STATIC_SCRATCH_BYTES];

namespace {

// Grid cap of the static entry point: 8 waves on each of up to 512 CUs (an MI355X launch uses
// 2048).  It bounds the partial slots, so that the BASELINE decode shapes fit the scratch array.
constexpr int kStaticMaxWaves = 4096;
constexpr int kMaxDevices = 64;

// Address of `scratch` on the current device, looked up once per device; nullptr on failure.
void *static_scratch() {
  static std::atomic<void *> addr[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  void *p = addr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) {
      (void)hipGetLastError();
      return nullptr;
    }
    addr[dev].store(p, std::memory_order_release);
  }
  return p;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool dtype_ok(int dtype) { return dtype == IC_DTYPE_BF16 || dtype == IC_DTYPE_F16 || dtype == IC_DTYPE_F32; }

// A stride (elements) keeps 16-byte chunks aligned when stride*elem % 16 == 0.
bool stride16(int64_t stride, int es) { return ((stride * es) & 15) == 0; }

int check_pool(int64_t sb, int64_t sh, int64_t st, int gn, int hd, int block_size, int64_t num_blocks,
               int es) {
  if (gn <= 0 || hd <= 0 || block_size <= 0 || num_blocks <= 0) return IC_ERR_BAD_SHAPE;
  if (sb <= 0 || sh <= 0 || st < hd) return IC_ERR_BAD_SHAPE;
  if ((hd * es) % 16 != 0) return IC_ERR_UNSUPPORTED;
  if (!stride16(sb, es) || !stride16(sh, es) || !stride16(st, es)) return IC_ERR_ALIGNMENT;
  return IC_OK;
}

int resolve_min_chunk(int min_chunk_tokens) {
  if (min_chunk_tokens == 0) min_chunk_tokens = ic::kDefaultMinChunkTokens;
  if (min_chunk_tokens < 16 || min_chunk_tokens % 16 != 0) return -1;
  return min_chunk_tokens;
}

// Both decode entry points and the variant on the library's own scratch: checks, then the launch.
// The workspace has partial slots for a grid of at most `max_waves` waves.
int decode_checked(void *out, int64_t out_stride_seq, const void *q, int64_t q_stride_seq,
                   const void *k_pool, const void *v_pool, int64_t pool_stride_block,
                   int64_t pool_stride_head, int64_t pool_stride_token, const int32_t *block_tables,
                   int64_t block_table_stride, const int32_t *context_lens, int n_seqs, int hn, int gn,
                   int hd, int block_size, int64_t num_blocks, int max_context_len, float scale,
                   int min_chunk_tokens, int cohort_size, const int32_t *cohort_shared_blocks,
                   void *workspace, size_t workspace_bytes, int max_waves, int dtype, void *stream,
                   const uint8_t *key_mask = nullptr, int64_t key_mask_stride_seq = 0,
                   int64_t key_mask_stride_head = 0, const ic::AppendRows *rows = nullptr) {
  if (n_seqs < 0 || hn <= 0 || gn <= 0 || hn % gn != 0 || max_context_len < 0 || cohort_size < 1)
    return IC_ERR_BAD_SHAPE;
  if (key_mask != nullptr) {
    if (dtype != IC_DTYPE_F32 || cohort_size != 1) return IC_ERR_UNSUPPORTED;
    if (key_mask_stride_seq < max_context_len || key_mask_stride_head < 0) return IC_ERR_BAD_SHAPE;
  }
  if (!dtype_ok(dtype)) return IC_ERR_UNSUPPORTED;
  const int es = ic::elem_size(dtype);
  if (int rc = check_pool(pool_stride_block, pool_stride_head, pool_stride_token, gn, hd, block_size,
                          num_blocks, es))
    return rc;
  if (n_seqs == 0) return IC_OK;
  if (!out || !q || !k_pool || !v_pool || !block_tables || !context_lens) return IC_ERR_NULL_POINTER;
  if (cohort_size > 1) {
    if (!cohort_shared_blocks) return IC_ERR_NULL_POINTER;
    if (dtype == IC_DTYPE_F32 || !ic::decode_layout(n_seqs, hn, gn, cohort_size).ok) return IC_ERR_UNSUPPORTED;
  }
  if (out_stride_seq < (int64_t)hn * hd || q_stride_seq < (int64_t)hn * hd) return IC_ERR_BAD_SHAPE;
  if (max_context_len == 0) max_context_len = 1;  // all-empty batch: the reduce pass writes zeros
  const int mc = resolve_min_chunk(min_chunk_tokens);
  if (mc < 0) return IC_ERR_BAD_SHAPE;
  const int64_t need_blocks = ((int64_t)max_context_len + block_size - 1) / block_size;
  if (block_table_stride < need_blocks) return IC_ERR_BAD_SHAPE;
  if (!aligned16(q) || !aligned16(k_pool) || !aligned16(v_pool) || !stride16(q_stride_seq, es))
    return IC_ERR_ALIGNMENT;
  // the matrix-core kernel stores 8- or 16-byte pieces of output rows
  if (es == 2 && (!aligned16(out) || !stride16(out_stride_seq, es))) return IC_ERR_ALIGNMENT;
  const ic::DecodeWorkspace ws = ic::decode_workspace(n_seqs, hn, gn, hd, cohort_size, max_waves);
  if (rows != nullptr) {
    if (!rows->k_new || !rows->v_new || !rows->slots || (rows->cos_table != nullptr) != (rows->sin_table != nullptr) ||
        (rows->cos_table && !rows->positions))
      return IC_ERR_NULL_POINTER;
    if (rows->new_stride_token < (int64_t)gn * hd || (rows->cos_table && rows->table_rows <= 0)) return IC_ERR_BAD_SHAPE;
    if (!aligned16(rows->k_new) || !aligned16(rows->v_new) || !stride16(rows->new_stride_token, es) ||
        !aligned16(rows->cos_table) || !aligned16(rows->sin_table))
      return IC_ERR_ALIGNMENT;
  } else if (!workspace || workspace_bytes < ws.total() || (reinterpret_cast<uintptr_t>(workspace) & 255u))
    return IC_ERR_WORKSPACE;

  ic::DecodeArgs a;
  a.out = out;
  a.out_stride_seq = out_stride_seq;
  a.q = q;
  a.q_stride_seq = q_stride_seq;
  a.k_pool = k_pool;
  a.v_pool = v_pool;
  a.pool = {pool_stride_block, pool_stride_head, pool_stride_token, num_blocks, block_size};
  a.block_tables = block_tables;
  a.block_table_stride = block_table_stride;
  a.context_lens = context_lens;
  a.n_seqs = n_seqs;
  a.hn = hn;
  a.gn = gn;
  a.hd = hd;
  a.max_context_len = max_context_len;
  a.scale = scale;
  a.min_chunk_tokens = mc;
  char *wsp = static_cast<char *>(workspace);
  a.cum_blocks = reinterpret_cast<int32_t *>(wsp);
  a.part_ml = reinterpret_cast<float *>(wsp + ws.cum_bytes);
  a.part_acc = reinterpret_cast<float *>(wsp + ws.cum_bytes + ws.ml_bytes);
  a.shared_slot0 = (int64_t)ws.shared_slot0;
  a.cohort_size = cohort_size;
  a.cohort_shared_blocks = cohort_shared_blocks;
  a.max_waves = max_waves;
  a.key_mask = key_mask;
  a.key_mask_stride_seq = key_mask_stride_seq;
  a.key_mask_stride_head = key_mask_stride_head;
  a.dtype = dtype;
  a.rows = rows;
  return ic::launch_paged_decode(a, static_cast<hipStream_t>(stream));
}

ic_prefill_call prefill_call(void *out, int64_t out_stride_token, const void *q, int64_t q_stride_token,
                             const void *k_pool, const void *v_pool, int64_t pool_stride_block,
                             int64_t pool_stride_head, int64_t pool_stride_token, const int32_t *block_tables,
                             int64_t block_table_stride, const int32_t *context_lens, const int32_t *cu_seqlens_q,
                             int n_seqs, int max_chunk_len, int hn, int gn, int hd, int block_size,
                             int64_t num_blocks, float scale, int causal, int dtype) {
  ic_prefill_call c = {};
  c.out = out;
  c.out_stride_token = out_stride_token;
  c.q = q;
  c.q_stride_token = q_stride_token;
  c.k_pool = k_pool;
  c.v_pool = v_pool;
  c.pool_stride_block = pool_stride_block;
  c.pool_stride_head = pool_stride_head;
  c.pool_stride_token = pool_stride_token;
  c.block_tables = block_tables;
  c.block_table_stride = block_table_stride;
  c.context_lens = context_lens;
  c.cu_seqlens_q = cu_seqlens_q;
  c.n_seqs = n_seqs;
  c.max_chunk_len = max_chunk_len;
  c.hn = hn;
  c.gn = gn;
  c.hd = hd;
  c.block_size = block_size;
  c.num_blocks = num_blocks;
  c.scale = scale;
  c.causal = causal;
  c.dtype = dtype;
  return c;
}

int prefill_checked(const ic_prefill_call &c, const uint8_t *mask, int64_t mask_stride_seq, int64_t mask_stride_head,
                    int64_t mask_stride_row, int64_t mask_keys, void *stream) {
  if (c.n_seqs < 0 || c.max_chunk_len < 0 || c.hn <= 0 || c.gn <= 0 || c.hn % c.gn != 0) return IC_ERR_BAD_SHAPE;
  if (!dtype_ok(c.dtype)) return IC_ERR_UNSUPPORTED;
  const int es = ic::elem_size(c.dtype);
  if (int rc = check_pool(c.pool_stride_block, c.pool_stride_head, c.pool_stride_token, c.gn, c.hd, c.block_size,
                          c.num_blocks, es))
    return rc;
  if (c.n_seqs == 0 || c.max_chunk_len == 0) return IC_OK;
  if (!c.out || !c.q || !c.k_pool || !c.v_pool) return IC_ERR_NULL_POINTER;
  if (c.context_lens == nullptr) {  // equal sequences
    if (c.block_tables != nullptr || c.cu_seqlens_q != nullptr) return IC_ERR_NULL_POINTER;
    if (c.row_pitch < c.max_chunk_len || c.uniform_context < 0 || c.uniform_context > c.block_size ||
        c.n_seqs > c.num_blocks)
      return IC_ERR_BAD_SHAPE;
  } else {
    const bool equal_chunks = c.cu_seqlens_q == nullptr && c.row_pitch > 0;
    if (!c.block_tables || (!c.cu_seqlens_q && !equal_chunks)) return IC_ERR_NULL_POINTER;
    if (c.block_table_stride <= 0 || (!equal_chunks && c.row_pitch != 0)) return IC_ERR_BAD_SHAPE;
    if (equal_chunks && (c.row_pitch < c.max_chunk_len || c.rows != nullptr)) return IC_ERR_BAD_SHAPE;
  }
  if (c.mask_bits != nullptr) {
    if (c.mask_lists == nullptr) return IC_ERR_NULL_POINTER;
    if (c.context_lens != nullptr || c.causal || mask != nullptr || c.mask_plane_seq < 0 || c.mask_plane_head < 0)
      return IC_ERR_BAD_SHAPE;
  }
  if (c.rows != nullptr && (c.context_lens == nullptr || c.n_rows <= 0 || c.q_rows <= 0)) return IC_ERR_BAD_SHAPE;
  if (c.n_rows > 0x7fffffff || c.q_rows > 0x7fffffff || (c.row_pitch > 0 && c.row_pitch * c.n_seqs > 0x7fffffff))
    return IC_ERR_UNSUPPORTED;
  if (c.out_stride_token < (int64_t)c.hn * c.hd || c.q_stride_token < (int64_t)c.hn * c.hd) return IC_ERR_BAD_SHAPE;
  if (!aligned16(c.q) || !aligned16(c.out) || !aligned16(c.k_pool) || !aligned16(c.v_pool) ||
      !stride16(c.q_stride_token, es) || !stride16(c.out_stride_token, es))
    return IC_ERR_ALIGNMENT;
  if (c.positions != nullptr) {
    if (!c.cos_table || !c.sin_table) return IC_ERR_NULL_POINTER;
    if (c.table_rows <= 0) return IC_ERR_BAD_SHAPE;
    if (!aligned16(c.cos_table) || !aligned16(c.sin_table)) return IC_ERR_ALIGNMENT;
  }
  ic::PrefillArgs a;
  a.out = c.out;
  a.out_stride_token = c.out_stride_token;
  a.q = c.q;
  a.q_stride_token = c.q_stride_token;
  a.k_pool = c.k_pool;
  a.v_pool = c.v_pool;
  a.pool = {c.pool_stride_block, c.pool_stride_head, c.pool_stride_token, c.num_blocks, c.block_size};
  a.block_tables = c.block_tables;
  a.block_table_stride = c.block_table_stride;
  a.context_lens = c.context_lens;
  a.cu_seqlens_q = c.cu_seqlens_q;
  a.n_seqs = c.n_seqs;
  a.max_chunk_len = c.max_chunk_len;
  a.hn = c.hn;
  a.gn = c.gn;
  a.hd = c.hd;
  a.scale = c.scale;
  a.causal = c.causal;
  a.dtype = c.dtype;
  a.mask = mask;
  a.mask_stride_seq = mask_stride_seq;
  a.mask_stride_head = mask_stride_head;
  a.mask_stride_row = mask_stride_row;
  a.mask_keys = mask_keys;
  a.rows = c.rows;
  a.n_rows = (int)c.n_rows;
  a.q_rows = (int)c.q_rows;
  a.row_pitch = c.row_pitch;
  a.uniform_context = c.uniform_context;
  a.positions = c.positions;
  a.cos_table = c.cos_table;
  a.sin_table = c.sin_table;
  a.table_rows = c.table_rows;
  a.mask_bits = c.mask_bits;
  a.mask_lists = c.mask_lists;
  a.mask_plane_seq = c.mask_plane_seq;
  a.mask_plane_head = c.mask_plane_head;
  return ic::launch_paged_prefill(a, static_cast<hipStream_t>(stream));
}

}  // namespace

namespace ic {

int device_cu_count() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int n = cache[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1)
      n = 256;
    cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

}  // namespace ic

extern "C" {

int ic_version(void) { return 200; }

int64_t ic_decode_occupancy_queries(void) { return ic::decode::decode_occupancy_queries(); }

int64_t ic_mfma_probe(int iters, void *sink, void *stream) {
  if (sink == nullptr) return IC_ERR_NULL_POINTER;
  if (iters < 1 || iters > (1 << 24)) return IC_ERR_BAD_SHAPE;
  if ((reinterpret_cast<uintptr_t>(sink) & 3) != 0) return IC_ERR_ALIGNMENT;
  return ic::launch_mfma_probe(iters, sink, static_cast<hipStream_t>(stream));
}

const char *ic_error_string(int code) {
  switch (code) {
    case IC_OK: return "ok";
    case IC_ERR_NULL_POINTER: return "a required pointer is NULL";
    case IC_ERR_BAD_SHAPE: return "a size or stride is non-positive or inconsistent";
    case IC_ERR_UNSUPPORTED: return "no kernel built for this dtype / head_dim / group / block size";
    case IC_ERR_WORKSPACE: return "workspace missing, misaligned or too small";
    case IC_ERR_LAUNCH: return "kernel launch failed";
    case IC_ERR_ALIGNMENT: return "pointer or stride is not 16-byte aligned";
    case IC_ERR_STATIC_LIMIT:
      return "the batch needs more scratch than the library's static buffer holds (IC_STATIC_SCRATCH_BYTES); "
             "use ic_paged_decode with a caller-provided workspace";
    default: return "unknown error code";
  }
}

int ic_kv_append(const void *k_new, const void *v_new, int64_t new_stride_token, void *k_pool,
                 void *v_pool, int64_t pool_stride_block, int64_t pool_stride_head,
                 int64_t pool_stride_token, const int64_t *slot_mapping, int64_t n_tokens, int gn,
                 int hd, int block_size, int64_t num_blocks, int dtype, void *stream) {
  if (n_tokens < 0) return IC_ERR_BAD_SHAPE;
  if (!dtype_ok(dtype)) return IC_ERR_UNSUPPORTED;
  const int es = ic::elem_size(dtype);
  if (int rc = check_pool(pool_stride_block, pool_stride_head, pool_stride_token, gn, hd, block_size,
                          num_blocks, es))
    return rc;
  if (n_tokens == 0) return IC_OK;
  if (!k_new || !v_new || !k_pool || !v_pool || !slot_mapping) return IC_ERR_NULL_POINTER;
  if (new_stride_token < (int64_t)gn * hd) return IC_ERR_BAD_SHAPE;
  if (!aligned16(k_new) || !aligned16(v_new) || !aligned16(k_pool) || !aligned16(v_pool) ||
      !stride16(new_stride_token, es))
    return IC_ERR_ALIGNMENT;
  ic::AppendArgs a;
  a.k_new = k_new;
  a.v_new = v_new;
  a.new_stride_token = new_stride_token;
  a.k_pool = k_pool;
  a.v_pool = v_pool;
  a.pool = {pool_stride_block, pool_stride_head, pool_stride_token, num_blocks, block_size};
  a.slot_mapping = slot_mapping;
  a.n_tokens = n_tokens;
  a.gn = gn;
  a.hd = hd;
  a.dtype = dtype;
  return ic::launch_kv_append(a, static_cast<hipStream_t>(stream));
}

int ic_rope_kv_append_to(void *q_out, int64_t q_out_stride_token, const void *q, int64_t q_stride_token, int hn,
                         const void *k_new, const void *v_new,
                      int64_t new_stride_token, void *k_pool, void *v_pool, int64_t pool_stride_block,
                      int64_t pool_stride_head, int64_t pool_stride_token, const int64_t *slot_mapping,
                      const int32_t *positions, const float *cos_table, const float *sin_table,
                      int64_t table_rows, int64_t n_tokens, int gn, int hd, int block_size,
                      int64_t num_blocks, int dtype, void *stream) {
  if (n_tokens < 0 || table_rows <= 0 || hd <= 0 || hd % 2 != 0) return IC_ERR_BAD_SHAPE;
  if (!dtype_ok(dtype)) return IC_ERR_UNSUPPORTED;
  const int es = ic::elem_size(dtype);
  if ((hd * es) % 16 != 0) return IC_ERR_UNSUPPORTED;
  const bool has_kv = k_new != nullptr || v_new != nullptr;
  if (has_kv) {
    if (int rc = check_pool(pool_stride_block, pool_stride_head, pool_stride_token, gn, hd, block_size,
                            num_blocks, es))
      return rc;
  }
  if (q != nullptr && hn <= 0) return IC_ERR_BAD_SHAPE;
  if (n_tokens == 0) return IC_OK;
  if (!positions || !cos_table || !sin_table) return IC_ERR_NULL_POINTER;
  if (q == nullptr && !has_kv) return IC_ERR_NULL_POINTER;
  if (!aligned16(cos_table) || !aligned16(sin_table)) return IC_ERR_ALIGNMENT;
  if (q != nullptr) {
    if (q_out == nullptr) return IC_ERR_NULL_POINTER;
    if (q_stride_token < (int64_t)hn * hd || q_out_stride_token < (int64_t)hn * hd) return IC_ERR_BAD_SHAPE;
    if (!aligned16(q) || !stride16(q_stride_token, es) || !aligned16(q_out) || !stride16(q_out_stride_token, es))
      return IC_ERR_ALIGNMENT;
  }
  if (has_kv) {
    if (!k_new || !v_new || !k_pool || !v_pool || !slot_mapping) return IC_ERR_NULL_POINTER;
    if (new_stride_token < (int64_t)gn * hd) return IC_ERR_BAD_SHAPE;
    if (!aligned16(k_new) || !aligned16(v_new) || !aligned16(k_pool) || !aligned16(v_pool) ||
        !stride16(new_stride_token, es))
      return IC_ERR_ALIGNMENT;
  }
  ic::RopeAppendArgs a;
  a.append.k_new = k_new;
  a.append.v_new = v_new;
  a.append.new_stride_token = new_stride_token;
  a.append.k_pool = k_pool;
  a.append.v_pool = v_pool;
  a.append.pool = {pool_stride_block, pool_stride_head, pool_stride_token, has_kv ? num_blocks : 0,
                   has_kv ? block_size : 1};
  a.append.slot_mapping = slot_mapping;
  a.append.n_tokens = n_tokens;
  a.append.gn = gn;
  a.append.hd = hd;
  a.append.dtype = dtype;
  a.q = q;
  a.q_stride_token = q_stride_token;
  a.q_out = q_out;
  a.q_out_stride_token = q_out_stride_token;
  a.hn = hn;
  a.positions = positions;
  a.cos_table = cos_table;
  a.sin_table = sin_table;
  a.table_rows = table_rows;
  return ic::launch_rope_kv_append(a, static_cast<hipStream_t>(stream));
}

int ic_rope_kv_append(void *q, int64_t q_stride_token, int hn, const void *k_new, const void *v_new,
                      int64_t new_stride_token, void *k_pool, void *v_pool, int64_t pool_stride_block,
                      int64_t pool_stride_head, int64_t pool_stride_token, const int64_t *slot_mapping,
                      const int32_t *positions, const float *cos_table, const float *sin_table,
                      int64_t table_rows, int64_t n_tokens, int gn, int hd, int block_size,
                      int64_t num_blocks, int dtype, void *stream) {
  return ic_rope_kv_append_to(q, q_stride_token, q, q_stride_token, hn, k_new, v_new, new_stride_token, k_pool, v_pool,
                              pool_stride_block, pool_stride_head, pool_stride_token, slot_mapping, positions,
                              cos_table, sin_table, table_rows, n_tokens, gn, hd, block_size, num_blocks, dtype,
                              stream);
}

size_t ic_paged_decode_workspace_bytes(int n_seqs, int hn, int gn, int hd) {
  return ic_paged_decode_shared_workspace_bytes(n_seqs, hn, gn, hd, 1);
}

size_t ic_paged_decode_shared_workspace_bytes(int n_seqs, int hn, int gn, int hd, int cohort_size) {
  if (n_seqs <= 0 || hn <= 0 || gn <= 0 || hn % gn != 0 || hd <= 0 || cohort_size < 1) return 0;
  if (!ic::decode_layout(n_seqs, hn, gn, cohort_size).ok) return 0;
  return ic::decode_workspace(n_seqs, hn, gn, hd, cohort_size).total();
}

int ic_paged_decode(void *out, int64_t out_stride_seq, const void *q, int64_t q_stride_seq,
                    const void *k_pool, const void *v_pool, int64_t pool_stride_block,
                    int64_t pool_stride_head, int64_t pool_stride_token, const int32_t *block_tables,
                    int64_t block_table_stride, const int32_t *context_lens, int n_seqs, int hn,
                    int gn, int hd, int block_size, int64_t num_blocks, int max_context_len,
                    float scale, int min_chunk_tokens, void *workspace, size_t workspace_bytes,
                    int dtype, void *stream) {
  return ic_paged_decode_shared(out, out_stride_seq, q, q_stride_seq, k_pool, v_pool, pool_stride_block,
                                pool_stride_head, pool_stride_token, block_tables, block_table_stride,
                                context_lens, n_seqs, hn, gn, hd, block_size, num_blocks,
                                max_context_len, scale, min_chunk_tokens, 1, nullptr, workspace,
                                workspace_bytes, dtype, stream);
}

int ic_paged_decode_shared(void *out, int64_t out_stride_seq, const void *q, int64_t q_stride_seq,
                           const void *k_pool, const void *v_pool, int64_t pool_stride_block,
                           int64_t pool_stride_head, int64_t pool_stride_token,
                           const int32_t *block_tables, int64_t block_table_stride,
                           const int32_t *context_lens, int n_seqs, int hn, int gn, int hd,
                           int block_size, int64_t num_blocks, int max_context_len, float scale,
                           int min_chunk_tokens, int cohort_size, const int32_t *cohort_shared_blocks,
                           void *workspace, size_t workspace_bytes, int dtype, void *stream) {
  return decode_checked(out, out_stride_seq, q, q_stride_seq, k_pool, v_pool, pool_stride_block,
                        pool_stride_head, pool_stride_token, block_tables, block_table_stride,
                        context_lens, n_seqs, hn, gn, hd, block_size, num_blocks, max_context_len,
                        scale, min_chunk_tokens, cohort_size, cohort_shared_blocks, workspace,
                        workspace_bytes, ic::kMaxDecodeWaves, dtype, stream);
}

size_t ic_paged_decode_static_scratch_bytes(int n_seqs, int hn, int gn, int hd) {
  if (n_seqs <= 0 || hn <= 0 || gn <= 0 || hn % gn != 0 || hd <= 0) return 0;
  return ic::decode_workspace(n_seqs, hn, gn, hd, 1, kStaticMaxWaves).total();
}

int ic_paged_decode_static(void *out, int64_t out_stride_seq, const void *q, int64_t q_stride_seq,
                           const void *k_pool, const void *v_pool, int64_t pool_stride_block,
                           int64_t pool_stride_head, int64_t pool_stride_token,
                           const int32_t *block_tables, int64_t block_table_stride,
                           const int32_t *context_lens, int n_seqs, int hn, int gn, int hd,
                           int block_size, int64_t num_blocks, int max_context_len, float scale,
                           int min_chunk_tokens, int dtype, void *stream) {
  if (n_seqs < 0 || hn <= 0 || gn <= 0 || hn % gn != 0 || hd <= 0) return IC_ERR_BAD_SHAPE;
  size_t need = 0;
  if (n_seqs > 0) {
    need = ic_paged_decode_static_scratch_bytes(n_seqs, hn, gn, hd);
    if (need == 0 || need > (size_t)IC_STATIC_SCRATCH_BYTES) return IC_ERR_STATIC_LIMIT;
  }
  void *ws = n_seqs > 0 ? static_scratch() : nullptr;  // an empty batch launches nothing
  if (n_seqs > 0 && ws == nullptr) return IC_ERR_LAUNCH;
  // Nothing in the workspace has to start at zero: the main kernel writes the prefix sums and
  // every partial the reduce pass reads, so a previous call's leftovers are never looked at.
  return decode_checked(out, out_stride_seq, q, q_stride_seq, k_pool, v_pool, pool_stride_block,
                        pool_stride_head, pool_stride_token, block_tables, block_table_stride,
                        context_lens, n_seqs, hn, gn, hd, block_size, num_blocks, max_context_len,
                        scale, min_chunk_tokens, 1, nullptr, ws, (size_t)IC_STATIC_SCRATCH_BYTES,
                        kStaticMaxWaves, dtype, stream);
}

size_t ic_linear_rows_workspace_bytes(int m, int n, int k, int splits, int dtype) {
  if (m < 1 || m > IC_LINEAR_ROWS_MAX || n < 1 || k < 1 || !dtype_ok(dtype)) return 0;
  const int got = ic::linear_rows_splits(n, k, dtype, splits);
  return got > 1 ? (size_t)got * m * n * sizeof(float) : 0;
}

int ic_linear_rows(void *out, int64_t out_stride, const void *x, int64_t x_stride, const void *w, int64_t w_stride,
                   const void *bias, int m, int n, int k, int splits, void *workspace, size_t workspace_bytes,
                   int dtype, void *stream) {
  if (m < 0 || n < 0 || k <= 0 || splits < 0) return IC_ERR_BAD_SHAPE;
  if (!dtype_ok(dtype)) return IC_ERR_UNSUPPORTED;
  if (m == 0 || n == 0) return IC_OK;
  const int es = ic::elem_size(dtype), block = 16 / es;
  if (m > IC_LINEAR_ROWS_MAX || n % block != 0 || k % (4 * block) != 0) return IC_ERR_UNSUPPORTED;
  if (out_stride < n || x_stride < k || w_stride < n) return IC_ERR_BAD_SHAPE;
  if (!out || !x || !w) return IC_ERR_NULL_POINTER;
  if (!aligned16(out) || !aligned16(x) || !aligned16(w) || !stride16(out_stride, es) || !stride16(x_stride, es) ||
      !stride16(w_stride, es))
    return IC_ERR_ALIGNMENT;
  const size_t need = ic_linear_rows_workspace_bytes(m, n, k, splits, dtype);
  if (need > 0 && (!workspace || !aligned16(workspace))) return IC_ERR_WORKSPACE;
  if (workspace_bytes < need) return IC_ERR_WORKSPACE;
  ic::LinearArgs a;
  a.x = x, a.w = w, a.bias = bias, a.out = out;
  a.x_stride = x_stride, a.w_stride = w_stride, a.out_stride = out_stride;
  a.m = m, a.n = n, a.k = k, a.splits = splits, a.dtype = dtype, a.workspace = workspace;
  return ic::launch_linear_rows(a, static_cast<hipStream_t>(stream));
}

// Sizes and modes of a step linear, without its pointers (what the workspace depends on).
static int step_linear_sizes(const ic_step_linear_call &a) {
  if (a.m < 0 || a.n < 0 || a.n2 < 0 || a.k < 0 || a.splits < 0) return IC_ERR_BAD_SHAPE;
  if (!dtype_ok(a.dtype) || a.norm < IC_NORM_NONE || a.norm > IC_NORM_RMS || a.act < IC_ACT_NONE ||
      a.act > IC_ACT_SWIGLU || (a.tile_bytes != 0 && a.tile_bytes != 64 && a.tile_bytes != 128 && a.tile_bytes != 256))
    return IC_ERR_UNSUPPORTED;
  const int block = 16 / ic::elem_size(a.dtype);
  const bool gated = a.act >= IC_ACT_GLU, append = a.slot_mapping != nullptr;
  const bool rows = a.residual != nullptr || a.norm != IC_NORM_NONE;
  if (a.m > IC_LINEAR_ROWS_MAX || (int64_t)a.n + a.n2 > (1 << 30) || a.n % (gated ? 2 * block : block) != 0 ||
      a.n2 % block != 0 || a.k % (4 * block) != 0 || (a.n == 0 && a.n2 > 0) ||
      (append && (rows || a.act != IC_ACT_NONE)) || ((gated || rows) && a.n2 != 0) ||
      (rows && (a.act != IC_ACT_NONE || a.n > IC_STEP_LINEAR_ROW_MAX)))
    return IC_ERR_UNSUPPORTED;
  if (a.w == nullptr ? !rows : a.k == 0) return a.w == nullptr ? IC_ERR_NULL_POINTER : IC_ERR_BAD_SHAPE;
  return IC_OK;
}

size_t ic_step_linear_workspace_bytes(const ic_step_linear_call *call) {
  if (call == nullptr || call->m == 0 || call->n == 0 || step_linear_sizes(*call) != IC_OK) return 0;
  const ic::StepPlan plan = ic::step_linear_plan(*call);
  return plan.partial ? (size_t)plan.splits * call->m * ((size_t)call->n + call->n2) * sizeof(float) : 0;
}

int ic_step_linear(const ic_step_linear_call *call, void *stream) {
  if (call == nullptr) return IC_ERR_NULL_POINTER;
  const ic_step_linear_call &a = *call;
  if (const int rc = step_linear_sizes(a); rc != IC_OK) return rc;
  if (a.m == 0 || a.n == 0) return IC_OK;
  const int es = ic::elem_size(a.dtype);
  const bool append = a.slot_mapping != nullptr;
  const int64_t columns = a.act >= IC_ACT_GLU ? a.n / 2 : append ? (int64_t)a.hn * a.hd : (int64_t)a.n + a.n2;
  if ((a.out && a.out_stride < columns) || (a.w && (a.x_stride < a.k || a.w_stride < a.n)) ||
      (a.n2 > 0 && a.w2_stride < a.n2) || (a.residual && a.residual_stride < columns) ||
      (a.norm != IC_NORM_NONE && a.norm_out_stride < columns))
    return IC_ERR_BAD_SHAPE;
  if ((a.w && !a.x) || (a.n2 > 0 && !a.w2) || (!a.out && a.norm == IC_NORM_NONE) ||
      (a.norm != IC_NORM_NONE && (!a.norm_weight || !a.norm_out)))
    return IC_ERR_NULL_POINTER;
  auto whole = [&](const void *ptr, int64_t stride) { return ptr == nullptr || (aligned16(ptr) && stride16(stride, es)); };
  if (!whole(a.out, a.out_stride) || !whole(a.norm_out, a.norm_out_stride) || !whole(a.x, a.x_stride) ||
      !whole(a.w, a.w_stride) || !whole(a.w2, a.w2_stride) || !whole(a.residual, a.residual_stride) ||
      !whole(a.norm_weight, 0) || !whole(a.norm_bias, 0))
    return IC_ERR_ALIGNMENT;
  if (append) {
    if (a.hn <= 0 || a.gn <= 0 || a.hd <= 0 || a.hd % 2 != 0 || a.block_size <= 0 || a.num_blocks <= 0 ||
        ((int64_t)a.hn + 2 * a.gn) * a.hd != (int64_t)a.n + a.n2 || a.pool_stride_block <= 0 ||
        a.pool_stride_head <= 0 || a.pool_stride_token <= 0)
      return IC_ERR_BAD_SHAPE;
    if (!a.k_pool || !a.v_pool || (a.cos_table != nullptr) != (a.sin_table != nullptr) ||
        (a.cos_table && (!a.positions || a.table_rows <= 0)))
      return IC_ERR_NULL_POINTER;
    if (!aligned16(a.k_pool) || !aligned16(a.v_pool) || !stride16(a.pool_stride_block, es) ||
        !stride16(a.pool_stride_head, es) || !stride16(a.pool_stride_token, es))
      return IC_ERR_ALIGNMENT;
  }
  const size_t need = ic_step_linear_workspace_bytes(call);
  if (need > 0 && (!a.workspace || !aligned16(a.workspace) || a.workspace_bytes < need)) return IC_ERR_WORKSPACE;
  return ic::launch_step_linear(a, static_cast<hipStream_t>(stream));
}

static int step_stack_sizes(const ic_step_stack_call &a) {
  if (a.num_layers < 0 || a.m < 0 || a.d <= 0 || a.f <= 0 || a.hn <= 0 || a.gn <= 0 || a.hd <= 0 || a.block_size <= 0 ||
      a.workgroups < 0 || a.max_context_len < 0 || a.max_polls < 0)
    return IC_ERR_BAD_SHAPE;
  if (!dtype_ok(a.dtype) || a.norm < IC_NORM_NONE || a.norm > IC_NORM_RMS || a.act < IC_ACT_NONE || a.act > IC_ACT_SWIGLU)
    return IC_ERR_UNSUPPORTED;
  const int es = ic::elem_size(a.dtype), unit = 64 / es;
  if (a.num_layers > IC_STEP_STACK_LAYERS || a.m > IC_STEP_STACK_ROWS || a.d > 1024 || a.d % unit != 0 ||
      a.f % unit != 0 || a.f > (1 << 18) || a.hn > 4096 || a.hn % a.gn != 0 || a.hn / a.gn > 4 || (a.hd != 64 && a.hd != 128) ||
      a.block_size % 16 != 0 || a.max_context_len > 2048 || a.workgroups > 4096)
    return IC_ERR_UNSUPPORTED;
  return IC_OK;
}

size_t ic_step_stack_workspace_bytes(const ic_step_stack_call *call) {
  if (call == nullptr || call->m == 0 || call->num_layers == 0 || step_stack_sizes(*call) != IC_OK) return 0;
  return ic::step_stack_workspace_bytes(*call);
}

int ic_step_stack(const ic_step_stack_call *call, void *stream) {
  if (call == nullptr) return IC_ERR_NULL_POINTER;
  const ic_step_stack_call &a = *call;
  if (const int rc = step_stack_sizes(a); rc != IC_OK) return rc;
  if (a.m == 0 || a.num_layers == 0) return IC_OK;
  const int es = ic::elem_size(a.dtype);
  if (const int rc = check_pool(a.pool_stride_block, a.pool_stride_head, a.pool_stride_token, a.gn, a.hd, a.block_size,
                                a.num_blocks, es))
    return rc;
  if (a.pool_stride_token >= ((int64_t)1 << 32) / (16 * es)) return IC_ERR_UNSUPPORTED;  // (32-bit offsets in a tile of 16 tokens)
  if (a.num_blocks * (a.block_size / 16) >= (int64_t)1 << 31 ||
      a.block_table_stride < ((int64_t)a.max_context_len + a.block_size - 1) / a.block_size)
    return IC_ERR_BAD_SHAPE;
  if (!a.layers || !a.x || (!a.out && a.norm == IC_NORM_NONE) || (a.norm != IC_NORM_NONE && (!a.norm_weight || !a.norm_out)) ||
      !a.block_tables || !a.context_lens || !a.slot_mapping || (a.cos_table != nullptr) != (a.sin_table != nullptr) ||
      (a.cos_table && (!a.positions || a.table_rows <= 0)))
    return IC_ERR_NULL_POINTER;
  bool whole = aligned16(a.x) && aligned16(a.out) && aligned16(a.norm_out) && aligned16(a.norm_weight) &&
               aligned16(a.norm_bias);
  for (int i = 0; i < a.num_layers; ++i) {
    const ic_step_layer &l = a.layers[i];
    if (!l.input_norm_weight || !l.q_weight || !l.kv_weight || !l.proj_weight || !l.post_norm_weight || !l.up_weight ||
        !l.down_weight || !l.k_pool || !l.v_pool)
      return IC_ERR_NULL_POINTER;
    if (l.input_norm < IC_NORM_LAYER || l.input_norm > IC_NORM_RMS || l.post_norm < IC_NORM_LAYER || l.post_norm > IC_NORM_RMS)
      return IC_ERR_UNSUPPORTED;
    for (const void *ptr : {l.input_norm_weight, l.input_norm_bias, l.q_weight, l.q_bias, l.kv_weight, l.kv_bias, l.proj_weight,
                            l.proj_bias, l.post_norm_weight, l.post_norm_bias, l.up_weight, l.up_bias, l.down_weight,
                            l.down_bias, (const void *)l.k_pool, (const void *)l.v_pool})
      whole = whole && aligned16(ptr);
  }
  if (!whole) return IC_ERR_ALIGNMENT;
  if (!a.workspace || reinterpret_cast<uintptr_t>(a.workspace) % 256 != 0 ||
      a.workspace_bytes < ic::step_stack_workspace_bytes(a))
    return IC_ERR_WORKSPACE;
  return ic::launch_step_stack(a, static_cast<hipStream_t>(stream));
}

int32_t *ic_step_status(void) {
  static int32_t *const word = []() -> int32_t * {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;  // (no part of a graph that this thread may be capturing)
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return nullptr;
    void *p = nullptr;
    if (hipHostMalloc(&p, 64, hipHostMallocPortable) != hipSuccess) p = nullptr, (void)hipGetLastError();
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (p != nullptr) memset(p, 0, 64);
    return static_cast<int32_t *>(p);
  }();
  return word;
}

int ic_paged_decode_append(const ic_decode_append_call *call, void *stream) {
  if (call == nullptr) return IC_ERR_NULL_POINTER;
  const ic_decode_append_call &c = *call;
  const ic::AppendRows rows = {c.k_new,     c.v_new,     c.new_stride_token, c.slot_mapping,
                               c.positions, c.cos_table, c.sin_table,        c.table_rows};
  return decode_checked(c.out, c.out_stride_seq, c.q, c.q_stride_seq, c.k_pool, c.v_pool, c.pool_stride_block,
                        c.pool_stride_head, c.pool_stride_token, c.block_tables, c.block_table_stride, c.context_lens,
                        c.n_seqs, c.hn, c.gn, c.hd, c.block_size, c.num_blocks, c.max_context_len, c.scale, 0, 1,
                        nullptr, nullptr, 0, ic::kMaxDecodeWaves, c.dtype, stream, nullptr, 0, 0, &rows);
}

size_t ic_greedy_workspace_bytes(int rows, int n) { return rows > 0 && n > 0 ? ic::greedy_workspace_bytes(rows, n) : 0; }

int ic_greedy(const ic_greedy_call *call, void *stream) {
  if (call == nullptr) return IC_ERR_NULL_POINTER;
  const ic_greedy_call &a = *call;
  if (a.rows < 0 || a.n < 2 || a.stride < a.n || ((a.tokens || a.margins) && a.columns < 1) ||
      (a.tokens && a.token_stride < a.columns) || (a.margins && a.margin_stride < a.columns))
    return IC_ERR_BAD_SHAPE;
  if (!dtype_ok(a.dtype)) return IC_ERR_UNSUPPORTED;
  if (a.rows == 0) return IC_OK;
  const int es = ic::elem_size(a.dtype);
  if (!a.logits) return IC_ERR_NULL_POINTER;
  if (!aligned16(a.logits) || !stride16(a.stride, es) || !stride16(a.n, es)) return IC_ERR_ALIGNMENT;
  if (!a.workspace || !aligned16(a.workspace) || a.workspace_bytes < ic_greedy_workspace_bytes(a.rows, a.n))
    return IC_ERR_WORKSPACE;
  return ic::launch_greedy(a, static_cast<hipStream_t>(stream));
}

int ic_advance(const ic_advance_call *call, void *stream) {
  if (call == nullptr) return IC_ERR_NULL_POINTER;
  const ic_advance_call &a = *call;
  if (a.rows < 0 || a.table_width < 0 || a.block_size < 1 || a.block_table_stride < a.table_width) return IC_ERR_BAD_SHAPE;
  if (a.rows == 0) return IC_OK;
  if (!a.context_lens || !a.block_tables || !a.positions || !a.token_positions || !a.slot_mapping)
    return IC_ERR_NULL_POINTER;
  return ic::launch_advance(a, static_cast<hipStream_t>(stream));
}

int ic_mask_pack(const uint8_t *mask, int64_t stride_seq, int64_t stride_head, int64_t stride_row, int n_seqs,
                 int heads, int rows, int keys, uint64_t *bits, int32_t *lists, int32_t *flags, void *stream) {
  if (n_seqs < 0 || heads < 0 || rows < 0 || keys < 0 || stride_seq < 0 || stride_head < 0 || stride_row < 0)
    return IC_ERR_BAD_SHAPE;
  if (n_seqs == 0 || heads == 0 || rows == 0 || keys == 0) return IC_OK;
  if (!mask || !bits || !lists || !flags) return IC_ERR_NULL_POINTER;
  return ic::launch_mask_pack(mask, stride_seq, stride_head, stride_row, n_seqs, heads, rows, keys, bits, lists, flags,
                              static_cast<hipStream_t>(stream));
}

// Rows to zero, checked; `empty`: nothing to do.
static int zero_rows(void *out, int64_t out_stride_bytes, int row_bytes, const int64_t *rows, int64_t n_rows,
                     const int32_t *bounds, int n_seqs, int row_pitch, ic::ZeroRows &z) {
  if (n_seqs < 0 || row_pitch < 0 || row_bytes <= 0 || n_rows < 0 || out_stride_bytes < row_bytes)
    return IC_ERR_BAD_SHAPE;
  if (n_seqs == 0 || row_pitch == 0) return IC_OK;
  if (!out || !bounds) return IC_ERR_NULL_POINTER;
  if (!aligned16(out) || out_stride_bytes % 16 != 0 || row_bytes % 16 != 0) return IC_ERR_ALIGNMENT;
  z.out = static_cast<char *>(out), z.stride_bytes = out_stride_bytes, z.chunks = row_bytes / 16;
  z.rows = rows, z.n_rows = n_rows, z.bounds = bounds;
  z.total = (int64_t)n_seqs * row_pitch, z.row_pitch = row_pitch;
  return IC_OK;
}

int ic_zero_unlisted_rows(void *out, int64_t out_stride_bytes, int row_bytes, const int64_t *rows, int64_t n_rows,
                          const int32_t *bounds, int n_seqs, int row_pitch, void *stream) {
  ic::ZeroRows z;
  if (n_seqs > 0 && row_pitch > 0 && out && !rows) return IC_ERR_NULL_POINTER;
  if (const int rc = zero_rows(out, out_stride_bytes, row_bytes, rows, n_rows, bounds, n_seqs, row_pitch, z); rc != IC_OK)
    return rc;
  return z.total == 0 ? IC_OK : ic::launch_zero_unlisted_rows(z, static_cast<hipStream_t>(stream));
}

int ic_append_chunks(const ic_append_call *call, void *stream) {
  if (call == nullptr) return IC_ERR_NULL_POINTER;
  const ic_append_call &c = *call;
  if (c.n_tokens < 0 || c.hd <= 0 || c.hd % 2 != 0 || (c.cos_table && c.table_rows <= 0)) return IC_ERR_BAD_SHAPE;
  if (!dtype_ok(c.dtype)) return IC_ERR_UNSUPPORTED;
  const int es = ic::elem_size(c.dtype);
  if (const int rc = check_pool(c.pool_stride_block, c.pool_stride_head, c.pool_stride_token, c.gn, c.hd, c.block_size,
                                c.num_blocks, es))
    return rc;
  ic::RopeAppendArgs a = {};
  if (c.zero_out != nullptr || c.rows != nullptr) {  // rows to zero, also where no token is appended or no row is listed
    if (c.rows == nullptr && c.n_rows != 0) return IC_ERR_NULL_POINTER;
    const int rc = zero_rows(c.zero_out, c.zero_stride_bytes, c.zero_row_bytes, c.rows, c.n_rows, c.bounds, c.n_seqs,
                             c.row_pitch, a.append.zero);
    if (rc != IC_OK) return rc;
  }
  if (c.n_tokens == 0)
    return a.append.zero.total == 0 ? IC_OK : ic::launch_zero_unlisted_rows(a.append.zero, static_cast<hipStream_t>(stream));
  if (!c.k_new || !c.v_new || !c.k_pool || !c.v_pool || !c.slot_mapping ||
      (c.cos_table != nullptr) != (c.sin_table != nullptr) || (c.cos_table && !c.positions))
    return IC_ERR_NULL_POINTER;
  if (c.new_stride_token < (int64_t)c.gn * c.hd) return IC_ERR_BAD_SHAPE;
  if (!aligned16(c.k_new) || !aligned16(c.v_new) || !aligned16(c.k_pool) || !aligned16(c.v_pool) ||
      !stride16(c.new_stride_token, es) || !aligned16(c.cos_table) || !aligned16(c.sin_table))
    return IC_ERR_ALIGNMENT;
  a.append.k_new = c.k_new, a.append.v_new = c.v_new, a.append.new_stride_token = c.new_stride_token;
  a.append.k_pool = c.k_pool, a.append.v_pool = c.v_pool;
  a.append.pool = {c.pool_stride_block, c.pool_stride_head, c.pool_stride_token, c.num_blocks, c.block_size};
  a.append.slot_mapping = c.slot_mapping, a.append.n_tokens = c.n_tokens;
  a.append.gn = c.gn, a.append.hd = c.hd, a.append.dtype = c.dtype;
  if (c.cos_table == nullptr) return ic::launch_kv_append(a.append, static_cast<hipStream_t>(stream));
  a.positions = c.positions, a.cos_table = c.cos_table, a.sin_table = c.sin_table, a.table_rows = c.table_rows;
  return ic::launch_rope_kv_append(a, static_cast<hipStream_t>(stream));
}

int ic_paged_prefill_ex(const ic_prefill_call *call, void *stream) {
  if (call == nullptr) return IC_ERR_NULL_POINTER;
  return prefill_checked(*call, nullptr, 0, 0, 0, 0, stream);
}

int ic_paged_prefill(void *out, int64_t out_stride_token, const void *q, int64_t q_stride_token,
                     const void *k_pool, const void *v_pool, int64_t pool_stride_block,
                     int64_t pool_stride_head, int64_t pool_stride_token,
                     const int32_t *block_tables, int64_t block_table_stride,
                     const int32_t *context_lens, const int32_t *cu_seqlens_q, int n_seqs,
                     int max_chunk_len, int hn, int gn, int hd, int block_size, int64_t num_blocks,
                     float scale, int causal, int dtype, void *stream) {
  const ic_prefill_call c = prefill_call(out, out_stride_token, q, q_stride_token, k_pool, v_pool, pool_stride_block,
                                         pool_stride_head, pool_stride_token, block_tables, block_table_stride,
                                         context_lens, cu_seqlens_q, n_seqs, max_chunk_len, hn, gn, hd, block_size,
                                         num_blocks, scale, causal, dtype);
  // (a null array is an error here: equal sequences are the descriptor call's)
  if (n_seqs > 0 && max_chunk_len > 0 && (!block_tables || !context_lens || !cu_seqlens_q)) return IC_ERR_NULL_POINTER;
  return prefill_checked(c, nullptr, 0, 0, 0, 0, stream);
}

int ic_paged_prefill_masked(void *out, int64_t out_stride_token, const void *q, int64_t q_stride_token,
                            const void *k_pool, const void *v_pool, int64_t pool_stride_block,
                            int64_t pool_stride_head, int64_t pool_stride_token,
                            const int32_t *block_tables, int64_t block_table_stride,
                            const int32_t *context_lens, const int32_t *cu_seqlens_q, int n_seqs,
                            int max_chunk_len, int hn, int gn, int hd, int block_size,
                            int64_t num_blocks, float scale, const uint8_t *mask,
                            int64_t mask_stride_seq, int64_t mask_stride_head, int64_t mask_stride_row,
                            int64_t mask_keys, int dtype, void *stream) {
  if (n_seqs > 0 && max_chunk_len > 0 && mask == nullptr) return IC_ERR_NULL_POINTER;
  if (mask_stride_seq < 0 || mask_stride_head < 0 || mask_stride_row < 0 || mask_keys < 0) return IC_ERR_BAD_SHAPE;
  if (mask_stride_row != 0 && mask_stride_row < mask_keys) return IC_ERR_BAD_SHAPE;
  if (n_seqs > 0 && max_chunk_len > 0 && mask_keys < 1) return IC_ERR_BAD_SHAPE;  // a mask row holds a byte at least
  const ic_prefill_call c = prefill_call(out, out_stride_token, q, q_stride_token, k_pool, v_pool, pool_stride_block,
                                         pool_stride_head, pool_stride_token, block_tables, block_table_stride,
                                         context_lens, cu_seqlens_q, n_seqs, max_chunk_len, hn, gn, hd, block_size,
                                         num_blocks, scale, 0, dtype);
  // (a null array is an error here: equal sequences are the descriptor call's)
  if (n_seqs > 0 && max_chunk_len > 0 && (!block_tables || !context_lens || !cu_seqlens_q)) return IC_ERR_NULL_POINTER;
  return prefill_checked(c, mask, mask_stride_seq, mask_stride_head, mask_stride_row, mask_keys, stream);
}

int ic_paged_decode_masked(void *out, int64_t out_stride_seq, const void *q, int64_t q_stride_seq,
                           const void *k_pool, const void *v_pool, int64_t pool_stride_block,
                           int64_t pool_stride_head, int64_t pool_stride_token,
                           const int32_t *block_tables, int64_t block_table_stride,
                           const int32_t *context_lens, int n_seqs, int hn, int gn, int hd,
                           int block_size, int64_t num_blocks, int max_context_len, float scale,
                           int min_chunk_tokens, const uint8_t *key_mask, int64_t key_mask_stride_seq,
                           int64_t key_mask_stride_head, void *workspace, size_t workspace_bytes,
                           int dtype, void *stream) {
  if (n_seqs > 0 && key_mask == nullptr) return IC_ERR_NULL_POINTER;
  return decode_checked(out, out_stride_seq, q, q_stride_seq, k_pool, v_pool, pool_stride_block,
                        pool_stride_head, pool_stride_token, block_tables, block_table_stride,
                        context_lens, n_seqs, hn, gn, hd, block_size, num_blocks, max_context_len,
                        scale, min_chunk_tokens, 1, nullptr, workspace, workspace_bytes,
                        ic::kMaxDecodeWaves, dtype, stream, key_mask, key_mask_stride_seq,
                        key_mask_stride_head);
}

}  // extern "C"
