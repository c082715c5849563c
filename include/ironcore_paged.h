/*
 * ironcore_paged.h -- C ABI of the MI355X (gfx950) paged-attention library.
 *
 * The reference (haanjack/ironcore) has no FFI, no KV cache and no native
 * code: its attention boundary is the Python call
 *     Attention.forward(query, key, value, attention_mask=None)
 *         ironcore/layers/attention.py:208-253
 * made from TransformerLayer.custom_forward
 *         ironcore/models/transformer.py:101-103
 * Each entry point below names the reference code whose work it takes over
 * when that call runs against a block KV cache.
 *
 * Conventions
 *  - Every pointer is a DEVICE pointer borrowed for the duration of the call
 *    (the kernels are enqueued on `stream`; the memory must stay valid until
 *    the stream reaches them).  The library never allocates or frees.
 *  - `stream` is a hipStream_t passed as void* (NULL = the default stream).
 *  - Return value: IC_OK (0) or a negative IC_ERR_* code.  Argument errors
 *    are detected on the host before anything is launched.  The library
 *    never throws and never exits the process.  Calls may come from any
 *    host thread; ordering is the stream's.  What the library remembers
 *    between calls never shows in a result: per device, the CU count and
 *    the address of the static scratch below; per process, the occupancy
 *    the runtime reported for each decode kernel variant and LDS size
 *    class (asked once, see ic_decode_occupancy_queries) and whether a
 *    variant's dynamic-LDS limit has been raised.  All of it is written
 *    once and read with atomics.
 *  - Host memory the library owns: the word of ic_step_status.
 *  - Device memory the library owns: one array of IC_STATIC_SCRATCH_BYTES
 *    (32 MiB), part of the code object, so every process that loads the
 *    library holds it on each GPU it uses, whether or not it ever calls
 *    ic_paged_decode_static (the only entry point that touches it).
 *  - Head dimensions with attention kernels: 32, 64 and 128 (the append
 *    entry points take any head dimension whose rows are a multiple of 16
 *    bytes); others return IC_ERR_UNSUPPORTED.  Block sizes: any multiple
 *    of 16 tokens.
 *  - Element type is selected by `dtype` (IC_DTYPE_*).  Strides are in
 *    ELEMENTS.  The head dimension is always contiguous.
 *
 * Block KV cache layout (defined by this library; the reference has none)
 *  - k_pool, v_pool: num_blocks blocks of `block_size` tokens.  Element
 *    (block, kv_head, token_in_block, d) lives at
 *        block*pool_stride_block + kv_head*pool_stride_head
 *        + token_in_block*pool_stride_token + d.
 *    The native layout is [num_blocks, gn, block_size, hd] contiguous
 *    (pool_stride_block = gn*block_size*hd, pool_stride_head = block_size*hd,
 *    pool_stride_token = hd), which makes one (block, kv_head) tile a single
 *    contiguous run of block_size*hd elements.
 *  - block_tables: int32 [n_seqs, block_table_stride]; entry j of row i is
 *    the pool block that holds tokens [j*block_size, (j+1)*block_size) of
 *    sequence i.  Rows may alias blocks (shared prefixes).
 *  - context_lens: int32 [n_seqs]; number of tokens visible to the query,
 *    including tokens appended for this step.
 *  - slot_mapping: int64 [n_tokens]; block*block_size + token_in_block for
 *    each new K/V row; a negative slot marks a padding row and is skipped.
 *  - GQA: query head h reads KV head h / (hn / gn)
 *    (ironcore/layers/attention.py:95-102).
 */
#ifndef IRONCORE_PAGED_H
#define IRONCORE_PAGED_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define IC_OK                 0
#define IC_ERR_NULL_POINTER  (-1)  /* a required pointer is NULL                 */
#define IC_ERR_BAD_SHAPE     (-2)  /* a size/stride is non-positive or inconsistent */
#define IC_ERR_UNSUPPORTED   (-3)  /* dtype / head_dim / group size / block size not built */
#define IC_ERR_WORKSPACE     (-4)  /* workspace missing or too small             */
#define IC_ERR_LAUNCH        (-5)  /* hipGetLastError() reported a launch failure */
#define IC_ERR_ALIGNMENT     (-6)  /* a pointer or stride breaks the 16-byte rule */
#define IC_ERR_STATIC_LIMIT  (-7)  /* batch too large for ic_paged_decode_static's scratch */

#define IC_DTYPE_BF16 0
#define IC_DTYPE_F16  1
#define IC_DTYPE_F32  2

/* Library ABI version (major*10000 + minor*100 + patch). */
int ic_version(void);

/* Static, NUL-terminated description of an IC_* code. */
const char *ic_error_string(int code);

/*
 * Diagnostic, no counterpart in the reference: launches a loop of `iters` x 16
 * independent v_mfma_f32_32x32x16_bf16 per wave, one wave per SIMD on every
 * CU, operands in registers (no memory, LDS or vector work), and returns the
 * launch's flop count (negative: IC_ERR_*).  Timed over a second or more of
 * back-to-back launches it gives the matrix rate the device sustains once its
 * clock has settled under load, which bench.py reports beside the nominal
 * 2.5 PFLOP/s.  sink: 4 bytes of device memory, never written in practice.
 */
int64_t ic_mfma_probe(int iters, void *sink, void *stream);

/*
 * Diagnostic, no counterpart in the reference: how many times the decode
 * launcher has asked the HIP runtime for a kernel's occupancy in this process.
 * The answers are kept per kernel variant and LDS size class (whole KiB), so
 * the count stops growing once a serving loop has seen its batch-size classes;
 * a launch whose answer is known makes no runtime query, which is what lets a
 * stream capture on any host thread follow a warm-up on another.
 */
int64_t ic_decode_occupancy_queries(void);

/*
 * KV append: copy the K/V rows a transformer layer produced for n_tokens new
 * tokens into their cache slots, bit for bit.  Replaces nothing in the
 * reference (which recomputes K/V for the whole sequence every step,
 * examples/generate_text.py:27); the rows are the `key`/`value` tensors of
 * ironcore/models/transformer.py:88-98.
 *
 *   k_new, v_new   [n_tokens, gn, hd], row stride new_stride_token, heads and
 *                  head_dim contiguous within a row
 *   slot_mapping   int64 [n_tokens]
 * Slots outside [0, num_blocks*block_size) are skipped.
 */
int ic_kv_append(const void *k_new, const void *v_new, int64_t new_stride_token,
                 void *k_pool, void *v_pool,
                 int64_t pool_stride_block, int64_t pool_stride_head,
                 int64_t pool_stride_token,
                 const int64_t *slot_mapping, int64_t n_tokens,
                 int gn, int hd, int block_size, int64_t num_blocks,
                 int dtype, void *stream);

/*
 * KV append with rotary position embedding: in one pass, rotate the query rows
 * in place, rotate the new key rows into their cache slots and copy the new
 * value rows into theirs.  Takes over ironcore/models/transformer.py:95-98
 * (query = rope(query); key = rope(key)) together with the append above.
 * Element pairs (2i, 2i+1) are rotated by the angle of table row
 * positions[t], with the arithmetic of
 * ironcore/layers/positional_embedding/rotary.py:69-83 (fp32, each product and
 * sum rounded separately, result rounded to the element type), so the result
 * is bit-identical to that expression evaluated by torch.
 *
 *   q              [n_tokens, hn, hd], row stride q_stride_token; rotated IN
 *                  PLACE; NULL = no query work
 *   k_new, v_new   as for ic_kv_append; both NULL = rotate q only (then the
 *                  pool arguments and slot_mapping are ignored)
 *   positions      int32 [n_tokens]: table row of each token, clamped to
 *                  [0, table_rows).  The reference indexes its tables by the
 *                  BATCH index of a row (rotary.py:55-64 after the transpose at
 *                  :55); a cached decoder passes the token's position in its
 *                  sequence.  The choice is the caller's.
 *   cos_table, sin_table   fp32 [table_rows, hd/2], 16-byte aligned: the
 *                  cos_emb / sin_emb buffers of rotary.py:36-51
 */
int ic_rope_kv_append(void *q, int64_t q_stride_token, int hn,
                      const void *k_new, const void *v_new, int64_t new_stride_token,
                      void *k_pool, void *v_pool,
                      int64_t pool_stride_block, int64_t pool_stride_head,
                      int64_t pool_stride_token,
                      const int64_t *slot_mapping, const int32_t *positions,
                      const float *cos_table, const float *sin_table, int64_t table_rows,
                      int64_t n_tokens, int gn, int hd, int block_size,
                      int64_t num_blocks, int dtype, void *stream);

/*
 * The same with the rotated query rows going to a buffer of their own (q_out,
 * row stride q_out_stride_token) instead of over the query; q_out == q is the
 * call above.
 */
int ic_rope_kv_append_to(void *q_out, int64_t q_out_stride_token,
                         const void *q, int64_t q_stride_token, int hn,
                         const void *k_new, const void *v_new, int64_t new_stride_token,
                         void *k_pool, void *v_pool,
                         int64_t pool_stride_block, int64_t pool_stride_head,
                         int64_t pool_stride_token,
                         const int64_t *slot_mapping, const int32_t *positions,
                         const float *cos_table, const float *sin_table, int64_t table_rows,
                         int64_t n_tokens, int gn, int hd, int block_size,
                         int64_t num_blocks, int dtype, void *stream);

/*
 * Workspace the decode entry point needs (block-count prefix sums and
 * split-K partials), in bytes, for a batch of n_seqs sequences with these
 * head counts.  Returns 0 for invalid arguments.
 */
size_t ic_paged_decode_workspace_bytes(int n_seqs, int hn, int gn, int hd);

/*
 * Paged decode: one query token per sequence against the block KV cache.
 * Computes what ironcore/layers/attention.py:68-142 (_attention) returns for
 * sq = 1 on the rows the block table points at:
 *     out[i, h*hd + d] = sum_j softmax_j(q[i,h] . k[i,j,h/G] * scale) * v[i,j,h/G,d]
 *
 *   out           [n_seqs, hn*hd], row stride out_stride_seq (16-byte aligned
 *                 rows for bf16 / fp16)
 *   q             [n_seqs, hn, hd], row stride q_stride_seq
 *   scale         multiplies q.k (the reference divides by sqrt(hd),
 *                 attention.py:65,110; pass 1/sqrt(hd))
 *   max_context_len  upper bound on context_lens; larger entries are clamped
 *                 to it, and block_table_stride must cover it
 *   min_chunk_tokens  the K/V stream of the whole batch is cut into equal
 *                 shares, one per resident wave (split-K); this is the
 *                 smallest share (multiple of 16), 0 = default
 *   block_size    a multiple of 16 (the kernel loads whole 16-token tiles)
 *   workspace     at least ic_paged_decode_workspace_bytes(...) bytes, 256-byte
 *                 aligned; contents need not be initialised
 * Sequences with context_lens[i] <= 0 produce zeros.
 */
int ic_paged_decode(void *out, int64_t out_stride_seq,
                    const void *q, int64_t q_stride_seq,
                    const void *k_pool, const void *v_pool,
                    int64_t pool_stride_block, int64_t pool_stride_head,
                    int64_t pool_stride_token,
                    const int32_t *block_tables, int64_t block_table_stride,
                    const int32_t *context_lens,
                    int n_seqs, int hn, int gn, int hd, int block_size,
                    int64_t num_blocks, int max_context_len, float scale,
                    int min_chunk_tokens, void *workspace, size_t workspace_bytes,
                    int dtype, void *stream);

/*
 * Paged decode for batches whose sequences alias prefix blocks (sampling
 * several continuations of one prompt: the block tables of a group repeat the
 * prompt's blocks, as a fork of the block KV cache leaves them).  Same result
 * as ic_paged_decode on the same arguments; the aliased blocks are streamed
 * from HBM once per cohort instead of once per sequence.  The reference has
 * no counterpart (it has no KV cache; every sample recomputes its prompt,
 * examples/generate_text.py:27); the attention it must reproduce is still
 * ironcore/layers/attention.py:68-142.
 *
 *   cohort_size           S >= 1: sequences i*S .. i*S+S-1 of the batch form
 *                         cohort i (the last one may be short).  1 = no
 *                         sharing, identical to ic_paged_decode.
 *                         bf16 / fp16 only; hn / gn <= 16, and S at most
 *                         8 * (16 / (hn / gn)) (integer division): a wave
 *                         carries the heads of 16 / (hn / gn) members and up
 *                         to 8 waves of a workgroup share a cohort's tiles.
 *   cohort_shared_blocks  int32 [ceil(n_seqs / S)]: for each cohort, how many
 *                         leading block-table entries are the SAME pool block
 *                         in all its members' rows.  May under-state the
 *                         sharing (0 is always valid); must not over-state it.
 *                         Only blocks every member's context covers entirely
 *                         are treated as shared.  Ignored (may be NULL) when
 *                         cohort_size is 1.
 *   workspace             at least ic_paged_decode_shared_workspace_bytes(...)
 * Everything else as for ic_paged_decode.
 */
size_t ic_paged_decode_shared_workspace_bytes(int n_seqs, int hn, int gn, int hd,
                                              int cohort_size);
int ic_paged_decode_shared(void *out, int64_t out_stride_seq,
                           const void *q, int64_t q_stride_seq,
                           const void *k_pool, const void *v_pool,
                           int64_t pool_stride_block, int64_t pool_stride_head,
                           int64_t pool_stride_token,
                           const int32_t *block_tables, int64_t block_table_stride,
                           const int32_t *context_lens,
                           int n_seqs, int hn, int gn, int hd, int block_size,
                           int64_t num_blocks, int max_context_len, float scale,
                           int min_chunk_tokens,
                           int cohort_size, const int32_t *cohort_shared_blocks,
                           void *workspace, size_t workspace_bytes,
                           int dtype, void *stream);

/*
 * Paged decode that allocates nothing and takes no workspace: ic_paged_decode
 * with the workspace (row prefix sums and split-K partials) in a static device
 * array of IC_STATIC_SCRATCH_BYTES inside the library.  It has no counterpart
 * in the reference; it is for callers that cannot allocate device memory and
 * have no workspace to pass: code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc.  Same arguments, same kernels and same
 * result as ic_paged_decode (the grid is capped at 4096 waves, which no current
 * GPU exceeds).
 *
 *  - Limit: ic_paged_decode_static_scratch_bytes(n_seqs, hn, gn, hd) must not
 *    exceed IC_STATIC_SCRATCH_BYTES, else IC_ERR_STATIC_LIMIT and nothing is
 *    launched.  The need is 520 * (4096 + n_seqs * gn * ceil(G / 8)) * min(G, 8)
 *    bytes at hd 128 (G = hn / gn), plus 4 * (n_seqs + 2) rounded up to 256:
 *    21.3 MB for 128 sequences of 64 q / 8 kv heads, 22.4 MB for 512 sequences
 *    of 28 / 4 heads, 3.2 MB for 64 sequences of 32 / 32 heads.
 *  - Each GPU the library is used on holds the array from the first call on
 *    that device until the process ends.  The first call on a device looks the
 *    array's address up (hipGetSymbolAddress) and, like the first launch of any
 *    kernel variant, must not be made under stream capture.
 *  - Every call on a GPU uses that GPU's one array: calls that overlap in time
 *    on one GPU (two streams, two host threads) race on the partials.  Calls
 *    ordered on one stream are safe; nothing in the array has to be cleared
 *    between calls (each call writes every value it later reads).
 */
#define IC_STATIC_SCRATCH_BYTES (32u << 20)
size_t ic_paged_decode_static_scratch_bytes(int n_seqs, int hn, int gn, int hd);
int ic_paged_decode_static(void *out, int64_t out_stride_seq,
                           const void *q, int64_t q_stride_seq,
                           const void *k_pool, const void *v_pool,
                           int64_t pool_stride_block, int64_t pool_stride_head,
                           int64_t pool_stride_token,
                           const int32_t *block_tables, int64_t block_table_stride,
                           const int32_t *context_lens,
                           int n_seqs, int hn, int gn, int hd, int block_size,
                           int64_t num_blocks, int max_context_len, float scale,
                           int min_chunk_tokens, int dtype, void *stream);

/*
 * Chunked prefill against the block KV cache: each sequence brings a chunk of
 * new query tokens whose K/V rows are already appended; query row r of a
 * chunk of length C in a sequence of context length L sees keys
 * j <= (L - C) + r.  Computes what attention.py:68-142 returns for
 * sq = C, sk = L with the causal mask of ironcore/language_model.py:109-114
 * shifted by the cached prefix.  With causal = 0 every query row sees all L
 * keys (the reference's attention_mask=None case).  bf16 / fp16 pools run on
 * the 16-bit matrix-core kernel; fp32 pools on an fp32 kernel that keeps
 * every product, sum and probability in fp32.
 *
 *   out           [n_tokens, hn*hd], row stride out_stride_token
 *   q             [n_tokens, hn, hd], row stride q_stride_token; the chunk of
 *                 sequence i is rows cu_seqlens_q[i] .. cu_seqlens_q[i+1]-1
 *   cu_seqlens_q  int32 [n_seqs + 1]
 *   max_chunk_len upper bound on any chunk length (sizes the grid)
 * The 16-bit kernel addresses inside a pool block with 32 bits: a call whose
 * pool_stride_block, or pool_stride_token times the rows of a block, reaches
 * 2^31 elements (a block of 4 GiB) returns IC_ERR_UNSUPPORTED.
 */
int ic_paged_prefill(void *out, int64_t out_stride_token,
                     const void *q, int64_t q_stride_token,
                     const void *k_pool, const void *v_pool,
                     int64_t pool_stride_block, int64_t pool_stride_head,
                     int64_t pool_stride_token,
                     const int32_t *block_tables, int64_t block_table_stride,
                     const int32_t *context_lens, const int32_t *cu_seqlens_q,
                     int n_seqs, int max_chunk_len,
                     int hn, int gn, int hd, int block_size,
                     int64_t num_blocks, float scale, int causal,
                     int dtype, void *stream);

/*
 * Packs a byte mask (nonzero = visible; strides in bytes, key stride 1) of
 * n_seqs x heads planes of `rows` x `keys` for ic_paged_prefill_ex: one bit per key,
 * the list of 64-key tiles each 128-row query tile has to visit, and two flags.
 * It reads the mask once for all heads that share it and for every later call
 * that uses it.  No counterpart in the reference, which adds its fill value to
 * the whole score matrix (attention.py:115-117).
 *
 *   bits   uint64 [n_seqs*heads][ceil(rows/128)*4][ceil(keys/64)][32]
 *   lists  int32 [n_seqs*heads][ceil(rows/128)][ceil(keys/64) + 1]
 *   flags  int32 [2], set to nonzero by the caller; flags[0] is cleared when the
 *          mask hides a key, flags[1] when it is not the causal pattern
 *          (row r sees keys j <= (keys - rows) + r)
 * At most 524 288 keys, 65 535 heads and sequences (else IC_ERR_UNSUPPORTED).
 */
int ic_mask_pack(const uint8_t *mask, int64_t stride_seq, int64_t stride_head, int64_t stride_row,
                 int n_seqs, int heads, int rows, int keys,
                 uint64_t *bits, int32_t *lists, int32_t *flags, void *stream);

/*
 * Chunked prefill by descriptor: ic_paged_prefill (same fields, same meaning)
 * plus three forms of input that spare a caller passes over its tensors.
 * Clear the struct first; a field left zero is the plain call's behaviour.
 *
 *   rows, n_rows, q_rows
 *                    rows != NULL: row i of the packed chunks (cu_seqlens_q) is row
 *                    rows[i] of q and out, of q_rows rows; n_rows entries.  The other
 *                    rows of out are left alone (ic_zero_unlisted_rows).
 *   uniform_context  with context_lens, cu_seqlens_q and block_tables all NULL:
 *                    equal sequences.  Every context has this many keys, every
 *                    chunk max_chunk_len rows, row_pitch >= max_chunk_len apart, and
 *                    sequence i is pool block i (uniform_context <= block_size,
 *                    any block size): a dense [b, s, gn, hd] tensor as a pool.
 *                    With context_lens: no context is longer, 0 if the caller does not
 *                    know (the block tables' width then bounds them).  It chooses
 *                    between kernels and bounds nothing.
 *   row_pitch        with context_lens and block_tables, cu_seqlens_q and rows NULL:
 *                    chunks of max_chunk_len rows each, row_pitch >= max_chunk_len apart.
 *   positions, cos_table, sin_table, table_rows
 *                    positions != NULL: the query rows have NOT been rotated;
 *                    row r of q is rotated as it is loaded, by table row
 *                    positions[r], with the arithmetic and the rounding of
 *                    ic_rope_kv_append.  The keys in the pool are rotated already.
 *   mask_bits, mask_lists, mask_plane_seq, mask_plane_head
 *                    mask_bits != NULL: a general mask of max_chunk_len rows and
 *                    uniform_context keys, packed by ic_mask_pack (equal sequences
 *                    only, causal = 0); sequence i and head h use plane
 *                    i*mask_plane_seq + h*mask_plane_head of it.  Semantics of
 *                    ic_paged_prefill_masked.
 */
typedef struct ic_prefill_call {
  void *out;
  int64_t out_stride_token;
  const void *q;
  int64_t q_stride_token;
  const void *k_pool;
  const void *v_pool;
  int64_t pool_stride_block, pool_stride_head, pool_stride_token;
  const int32_t *block_tables;
  int64_t block_table_stride;
  const int32_t *context_lens;
  const int32_t *cu_seqlens_q;
  int n_seqs, max_chunk_len;
  int hn, gn, hd, block_size;
  int64_t num_blocks;
  float scale;
  int causal;
  int dtype;
  int uniform_context;
  int64_t row_pitch;
  const int64_t *rows;
  int64_t n_rows, q_rows;
  const int32_t *positions;
  const float *cos_table;
  const float *sin_table;
  int64_t table_rows;
  const uint64_t *mask_bits;
  const int32_t *mask_lists;
  int mask_plane_seq, mask_plane_head;
} ic_prefill_call;
int ic_paged_prefill_ex(const ic_prefill_call *call, void *stream);

/*
 * Zeroes rows of a padded output [n_seqs * row_pitch rows of row_bytes, 16-byte
 * aligned] ahead of a prefill call with `rows`: at least every row that is not
 * among rows[0 .. n_rows-1].  (A row that is listed anywhere but at its sequence's
 * start, entry bounds[i] + r for row i*row_pitch + r, may be zeroed too: the
 * attention call writes it afterwards.)
 */
int ic_zero_unlisted_rows(void *out, int64_t out_stride_bytes, int row_bytes, const int64_t *rows, int64_t n_rows,
                          const int32_t *bounds, int n_seqs, int row_pitch, void *stream);

/*
 * Chunked prefill under a general attention mask: ic_paged_prefill with the
 * causal rule replaced by the caller's mask, for the attention_mask argument
 * of ironcore/layers/attention.py:208-253 when it is neither absent nor the
 * causal pattern (any mask broadcastable to [b, 1, sq, sk], attention.py:115-117;
 * e.g. the per-document masks of ironcore/language_model.py:140-152).
 *
 *   mask    uint8; the byte of (sequence i, query head h, chunk row r, key j) is
 *           mask[i*mask_stride_seq + h*mask_stride_head + r*mask_stride_row + j],
 *           nonzero = visible.  A stride of 0 broadcasts over that index.
 *   mask_keys  keys every mask row covers (its extent along j): a key at or
 *           beyond it is hidden, and no byte past it is read.
 * Hidden keys get the reference's FINITE fill value (attention.py:66): next to a
 * visible key they weigh nothing; a query row with no visible key returns the
 * plain average of V over its context, as the reference does.  A chunk may be
 * longer than its context here (sq > sk).  bf16, fp16 and fp32.
 */
int ic_paged_prefill_masked(void *out, int64_t out_stride_token,
                            const void *q, int64_t q_stride_token,
                            const void *k_pool, const void *v_pool,
                            int64_t pool_stride_block, int64_t pool_stride_head,
                            int64_t pool_stride_token,
                            const int32_t *block_tables, int64_t block_table_stride,
                            const int32_t *context_lens, const int32_t *cu_seqlens_q,
                            int n_seqs, int max_chunk_len,
                            int hn, int gn, int hd, int block_size,
                            int64_t num_blocks, float scale,
                            const uint8_t *mask, int64_t mask_stride_seq,
                            int64_t mask_stride_head, int64_t mask_stride_row,
                            int64_t mask_keys, int dtype, void *stream);

/*
 * Paged decode under a key mask, fp32 only: ic_paged_decode where sequence i's
 * query head h sees key j only if
 * key_mask[i*key_mask_stride_seq + h*key_mask_stride_head + j] is nonzero
 * (key_mask_stride_head 0 = one mask row for all heads; key_mask_stride_seq
 * >= max_context_len).  Same finite-fill semantics as ic_paged_prefill_masked.
 * For single-token steps of an fp32 model under a general mask; chunks, and
 * 16-bit calls of any length, use ic_paged_prefill_masked (16-bit pools get
 * IC_ERR_UNSUPPORTED here).
 */
int ic_paged_decode_masked(void *out, int64_t out_stride_seq,
                           const void *q, int64_t q_stride_seq,
                           const void *k_pool, const void *v_pool,
                           int64_t pool_stride_block, int64_t pool_stride_head,
                           int64_t pool_stride_token,
                           const int32_t *block_tables, int64_t block_table_stride,
                           const int32_t *context_lens,
                           int n_seqs, int hn, int gn, int hd, int block_size,
                           int64_t num_blocks, int max_context_len, float scale,
                           int min_chunk_tokens,
                           const uint8_t *key_mask, int64_t key_mask_stride_seq,
                           int64_t key_mask_stride_head,
                           void *workspace, size_t workspace_bytes,
                           int dtype, void *stream);

/*
 * y = x W (+ bias) for at most IC_LINEAR_ROWS_MAX rows: the projections of a
 * decode step (the reference's linears, W stored [in, out]:
 * ironcore/parallel/tensor_parallel/layers.py:41,194-204).  fp32 sums.
 *
 *   out [m, n], x [m, k], w [k, n], bias [n] or NULL: one element type, rows
 *       16-byte aligned; strides in elements.
 *   n a multiple of 16 bytes of elements, k of 64 bytes.
 *   splits  workgroups that share a column's k range; 0 lets the library choose.
 *   workspace  ic_linear_rows_workspace_bytes(m, n, k, splits, dtype) bytes.
 */
#define IC_LINEAR_ROWS_MAX 32
size_t ic_linear_rows_workspace_bytes(int m, int n, int k, int splits, int dtype);
int ic_linear_rows(void *out, int64_t out_stride, const void *x, int64_t x_stride,
                   const void *w, int64_t w_stride, const void *bias,
                   int m, int n, int k, int splits,
                   void *workspace, size_t workspace_bytes, int dtype, void *stream);

/*
 * A linear of a decode step with what stands around it in a transformer layer
 * (ironcore/models/transformer.py:77-135), for at most IC_LINEAR_ROWS_MAX rows, in
 * one of three forms:
 *
 *   out = act(x W + bias)
 *   [q | k | v] = x W + bias, stored as an append   (slot_mapping not NULL)
 *   out = x W + bias + residual, norm_out = norm(out)   (residual or norm given)
 *
 * One element type throughout, fp32 sums, rounded to the element type only on
 * the way to out and norm_out (the norm takes out as rounded).  Rows of x, residual,
 * out, norm_out, w, w2, norm_weight and norm_bias 16-byte aligned, strides in elements;
 * k a multiple of 64 bytes of elements, n, n2 and half of a gated n of 16 bytes.
 *
 *   w2     a second matrix [k, n2] whose columns follow the first one's, or NULL
 *          (third form: NULL).
 *   act    IC_ACT_*, first form; the gated ones take the columns [feature | gate] and
 *          give n / 2: GLU feature * sigmoid(gate), SWIGLU silu(feature) * gate.
 *   slot_mapping  second form: the columns are hn heads of queries, gn of keys and gn
 *          of values (w and w2 together); queries go to out, keys and values into
 *          the pools as ic_kv_append stores them.  With cos_table and sin_table
 *          queries and keys are rotated on the way as by ic_rope_kv_append, row i at
 *          positions[i].
 *   norm   third form: IC_NORM_* over the n values of a row, weight [n], bias [n] or
 *          NULL; out may be NULL then.  With w NULL the product and the bias are left out.
 *          n up to IC_STEP_LINEAR_ROW_MAX.
 *   tile_bytes  64, 128 or 256: bytes of a row of W that a workgroup takes; splits:
 *          workgroups that share a column's k range; 0 lets the library choose.
 *   workspace  ic_step_linear_workspace_bytes(call) bytes, 16-byte aligned.
 */
enum { IC_NORM_NONE = 0, IC_NORM_LAYER = 1, IC_NORM_RMS = 2 };
enum { IC_ACT_NONE = 0, IC_ACT_RELU = 1, IC_ACT_GELU = 2, IC_ACT_SILU = 3, IC_ACT_GLU = 4, IC_ACT_SWIGLU = 5 };
#define IC_STEP_LINEAR_ROW_MAX 16384
typedef struct ic_step_linear_call {
  void *out, *norm_out;
  int64_t out_stride, norm_out_stride;
  const void *x;
  int64_t x_stride;
  const void *w, *bias;
  int64_t w_stride;
  const void *w2, *bias2;
  int64_t w2_stride;
  const void *residual;
  int64_t residual_stride;
  const void *norm_weight, *norm_bias;
  int m, k, n, n2;
  int norm, act;
  float eps;
  int dtype, tile_bytes, splits;
  void *k_pool, *v_pool;
  int64_t pool_stride_block, pool_stride_head, pool_stride_token, num_blocks;
  int hn, gn, hd, block_size;
  const int64_t *slot_mapping;
  const int32_t *positions;
  const float *cos_table, *sin_table;
  int64_t table_rows;
  void *workspace;
  size_t workspace_bytes;
} ic_step_linear_call;
size_t ic_step_linear_workspace_bytes(const ic_step_linear_call *call);
int ic_step_linear(const ic_step_linear_call *call, void *stream);

/*
 * All layers of a decode step in one launch, pre-LN, one new token a row: per layer the
 * norm, [q | k | v] = x W + bias (rotated with cos_table and sin_table, k and v appended as
 * by ic_kv_append), ic_paged_decode, output projection and residual, norm, up-projection
 * with the activation, down-projection and residual; then out (or NULL) = the last
 * layer's output and norm_out = its norm (norm IC_NORM_NONE: none, NULL).  Rounded to the element type
 * where ic_step_linear calls round.
 *
 * For small models and batches; everything else is IC_ERR_UNSUPPORTED with nothing launched:
 * m up to IC_STEP_STACK_ROWS, up to IC_STEP_STACK_LAYERS layers of one shape, d up to 1 024,
 * heads of 64 or 128, at most 4 query heads to a KV head, contexts up to 2 048
 * tokens.  Matrices [in, out] without gaps, 16-byte aligned; d, f, hn * hd and gn * hd
 * multiples of 64 bytes of elements.  up_weight has 2 f columns [feature | gate] with a gated act.
 *
 *   workspace  ic_step_stack_workspace_bytes(call) bytes, 256-byte aligned (0: unsupported).
 *   workgroups  0: one to a CU.  draw: nonzero deals the work by a counter, as the launch does
 *          by itself when other work keeps its workgroups from starting together.
 *   max_polls, status  a wait for another workgroup's results is given up after so many polls (0: 4 194 304,
 *          seconds; met only if a part of the launch stopped).  The launch then ends all the same: rows of out and
 *          norm_out that needed those results hold NaNs, no row that came of them is appended (rows of the step may be
 *          missing from the pools, none is wrong), and *status, if not NULL, is set to 1.  It is never cleared
 *          here; device or pinned host memory that lives until the launch has ended, such as ic_step_status().
 */
#define IC_STEP_STACK_LAYERS 16
#define IC_STEP_STACK_ROWS 16
typedef struct ic_step_layer {
  const void *input_norm_weight, *input_norm_bias;
  const void *q_weight, *q_bias, *kv_weight, *kv_bias;
  const void *proj_weight, *proj_bias;
  const void *post_norm_weight, *post_norm_bias;
  const void *up_weight, *up_bias, *down_weight, *down_bias;
  void *k_pool, *v_pool;
  int input_norm, post_norm;
  float input_norm_eps, post_norm_eps;
} ic_step_layer;
typedef struct ic_step_stack_call {
  const ic_step_layer *layers;
  const void *x;
  void *out, *norm_out;
  const void *norm_weight, *norm_bias;
  int num_layers, m, d, f, hn, gn, hd, act;
  int norm;
  float eps;
  int64_t pool_stride_block, pool_stride_head, pool_stride_token, num_blocks;
  const int32_t *block_tables;
  int64_t block_table_stride;
  const int32_t *context_lens;
  const int64_t *slot_mapping;
  const int32_t *positions;
  const float *cos_table, *sin_table;
  int64_t table_rows;
  int block_size, max_context_len;
  float scale;
  int dtype, workgroups, draw;
  void *workspace;
  size_t workspace_bytes;
  int32_t *status;
  int max_polls;
} ic_step_stack_call;
size_t ic_step_stack_workspace_bytes(const ic_step_stack_call *call);
int ic_step_stack(const ic_step_stack_call *call, void *stream);

/*
 * A word for `status` that launches in flight may write at any time: pinned host memory, one for the process, allocated
 * and cleared by the first call and never freed (NULL: not to be had).  The library neither reads it nor hands it to a
 * launch by itself.  Any host thread, also while a stream is capturing.
 */
int32_t *ic_step_status(void);

/*
 * The append of a step's chunks in one launch: ic_kv_append, or with cos_table and
 * sin_table ic_rope_kv_append_to without queries, and with zero_out not NULL
 * ic_zero_unlisted_rows (zero_out, zero_stride_bytes, zero_row_bytes, rows, n_rows, bounds,
 * n_seqs, row_pitch) beside it, also where there is no token to append (n_tokens 0) or no
 * row that a chunk holds (n_rows 0: rows may be NULL then).
 */
typedef struct ic_append_call {
  const void *k_new, *v_new;
  int64_t new_stride_token;
  void *k_pool, *v_pool;
  int64_t pool_stride_block, pool_stride_head, pool_stride_token, num_blocks;
  const int64_t *slot_mapping;
  int64_t n_tokens;
  int gn, hd, block_size, dtype;
  const int32_t *positions;
  const float *cos_table, *sin_table;
  int64_t table_rows;
  void *zero_out;
  int64_t zero_stride_bytes;
  const int64_t *rows;
  int64_t n_rows;
  const int32_t *bounds;
  int zero_row_bytes, n_seqs, row_pitch;
} ic_append_call;
int ic_append_chunks(const ic_append_call *call, void *stream);

/*
 * A decode step's append and attention in one launch: ic_kv_append (with cos_table and
 * sin_table ic_rope_kv_append_to, the query rows rotated on their way and not stored) of the
 * n_seqs new rows, then ic_paged_decode, which sees all of them, whichever sequence's
 * slot they are in.  For small batches of short contexts (at most 64 sequences, a KV
 * head of one to each CU, fewer where query heads share a KV head or contexts are longer);
 * IC_ERR_UNSUPPORTED for the others, with nothing launched.  No workspace.
 */
typedef struct ic_decode_append_call {
  void *out;
  int64_t out_stride_seq;
  const void *q;
  int64_t q_stride_seq;
  const void *k_new, *v_new;
  int64_t new_stride_token;
  void *k_pool, *v_pool;
  int64_t pool_stride_block, pool_stride_head, pool_stride_token, num_blocks;
  const int32_t *block_tables;
  int64_t block_table_stride;
  const int32_t *context_lens;
  const int64_t *slot_mapping;
  const int32_t *positions;
  const float *cos_table, *sin_table;
  int64_t table_rows;
  int n_seqs, hn, gn, hd, block_size, max_context_len;
  float scale;
  int dtype;
} ic_decode_append_call;
int ic_paged_decode_append(const ic_decode_append_call *call, void *stream);

/*
 * The next token of each row of logits, greedily (examples/generate_text.py:27-28 at
 * temperature 0): the first of the largest values, NaN counting as the largest.
 *
 *   logits [rows, n] of dtype, rows 16-byte aligned, n a multiple of 16 bytes and >= 2.
 *   tokens, margins  [rows, columns] or NULL: the token and best - second best (of
 *          equal values the second is as large as the best) go to column *column
 *          (NULL: 0); a column outside [0, columns) is not stored.
 *   next   [rows] or NULL: the token once more.
 *   finished  [rows] or NULL: a row with a nonzero byte gets eos, and a row whose
 *          token is eos gets a nonzero byte.
 *   workspace  ic_greedy_workspace_bytes(rows, n) bytes, 16-byte aligned.
 */
typedef struct ic_greedy_call {
  const void *logits;
  int64_t stride;
  int rows, n, dtype;
  int64_t *tokens;
  int64_t token_stride;
  float *margins;
  int64_t margin_stride;
  const int64_t *column;
  int64_t columns;
  int64_t *next;
  uint8_t *finished;
  int64_t eos;
  void *workspace;
  size_t workspace_bytes;
} ic_greedy_call;
size_t ic_greedy_workspace_bytes(int rows, int n);
int ic_greedy(const ic_greedy_call *call, void *stream);

/*
 * The bookkeeping of a decode step on the device: row i's new token has position
 * p = context_lens[i] (written to positions and token_positions), its pool slot is
 * block_tables[i][p / block_size] * block_size + p % block_size (-1 beyond
 * table_width), and context_lens[i] becomes p + 1.  *column (if given) grows by 1.
 */
typedef struct ic_advance_call {
  int32_t *context_lens;
  const int32_t *block_tables;
  int64_t block_table_stride;
  int rows, table_width, block_size;
  int32_t *positions;
  int64_t *token_positions;
  int64_t *slot_mapping;
  int64_t *column;
} ic_advance_call;
int ic_advance(const ic_advance_call *call, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* IRONCORE_PAGED_H */
