// Pieces shared by the chunked-prefill kernels (the 16-bit matrix-core kernel
// of paged_prefill.hip and the fp32 one of paged_prefill_f32.hip): kernel
// parameters, the values that stand for hidden scores, the exchange between a
// wave's two lane halves.
#pragma once

#include "ic_device.h"
#include "ic_internal.h"
#include "rope_device.h"

namespace ic {
namespace prefill {

struct PrefillKP {
  const char *q;
  const char *k_pool;
  const char *v_pool;
  const int32_t *block_tables;
  const int32_t *context_lens;
  const int32_t *cu_seqlens_q;
  char *out;
  int64_t q_stride_token;    // elements
  int64_t out_stride_token;  // elements
  int64_t stride_block;
  int64_t stride_head;
  int64_t stride_token;
  int64_t bt_stride;
  int64_t num_blocks;
  int block_size;   // a multiple of 16 tokens
  int block_shift;  // log2(block_size) when it is a power of two, else -1
  uint32_t block_magic;  // row / block_size == mulhi(row, block_magic): 2^32 / block_size for a power of two
                         // (exact for every row), else floor(2^32 / block_size) + 1 (exact below 2^32 / block_size)
  int group;        // query heads per KV head
  int gn;           // KV heads
  int n_units;      // n_seqs * gn
  int n_qtiles;     // query tiles per chunk (grid sizing); short kernel: workgroups per unit
  int by_sweep;     // short kernel: workgroups are numbered over all sequences, longest sweep first
  int flip_slice;   // short kernel: first slice of units whose workgroups take their blocks shortest sweep first
  int causal;
  float scale_log2e;
  // General attention mask (MASK variant): byte (sequence i, head h, chunk row r, key j) at
  // mask[i*mask_stride_seq + h*mask_stride_head + r*mask_stride_row + j], nonzero = visible.
  const uint8_t *mask;
  int64_t mask_stride_seq;
  int64_t mask_stride_head;
  int64_t mask_stride_row;
  int mask_keys;  // keys a mask row covers: keys from there on are hidden and never read
  const int64_t *rows;  // row of q and out that row i of the packed chunks is (nullptr: i itself)
  int n_rows;           // entries of `rows`
  int q_rows;           // rows of q and out, which bound them
  int64_t row_pitch;    // no cu_seqlens_q (equal chunks): rows from one chunk to the next in q and out
  int max_chunk;        // ... and rows of every chunk
  int uniform_context;  // context_lens == nullptr (equal sequences): keys of every context
  const int32_t *positions;  // rotary embedding of the query rows (nullptr: none)
  const float *cos_table;
  const float *sin_table;
  int table_rows;
  int half_hd;
  const uint64_t *mask_bits;   // packed mask: see mask_pack.hip
  const int32_t *mask_lists;
  int mask_plane_seq;
  int mask_plane_head;
  int mask_tiles;    // 64-key tiles of a mask row
  int mask_qtiles;   // 128-row query tiles of a plane
};

constexpr float kNegInf = -__builtin_huge_valf();
// Raw score of a key the mask hides.  The reference fills hidden scores with the FINITE minimum
// of the element type (attention.py:66,115-117), not -inf: beside any visible key the hidden ones
// get probability 0 either way, but a row with no visible key at all becomes a uniform average of
// V over the whole context.  A power of two, so that its product with the scale is exact and the
// exponent of a fully hidden row is exactly 0.
constexpr float kHiddenScore = -0x1p100f;

// x of this lane and x of lane ^ 32, as a pair (v_permlane32_swap: a vector-ALU
// exchange, where a shuffle would be an LDS operation and share its counter).
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void both_halves(float x, float &a, float &b) {
  const unsigned int u = __builtin_bit_cast(unsigned int, x);
  const u32x2_t r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  unsigned int r0 = r[0], r1 = r[1];
  // Opaque to the optimiser, which otherwise takes the two results of the swap
  // for the same value and folds max(r0, r1) to r0.
  asm("" : "+v"(r0), "+v"(r1));
  a = __builtin_bit_cast(float, r0);
  b = __builtin_bit_cast(float, r1);
}

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(8))) short s16x8_t;

// MFMA wrappers per element type: operands are 8 packed 16-bit values.
struct MmaBf16 {
  using E = Bf16;
  using T = __bf16;
  static __device__ __forceinline__ f32x16_t mma(const Vec16 &a, const Vec16 &b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    bf16x2_t v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
    return __builtin_bit_cast(uint32_t, v);
  }
};
struct MmaF16 {
  using E = F16;
  using T = _Float16;
  static __device__ __forceinline__ f32x16_t mma(const Vec16 &a, const Vec16 &b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    f16x2_t v = {static_cast<_Float16>(lo), static_cast<_Float16>(hi)};
    return __builtin_bit_cast(uint32_t, v);
  }
};

constexpr int kXcds = 8;

// An LDS tile is unpadded [token][dim], CPR 16-byte chunks to a row, and chunk c
// of row r lies in slot c ^ swizzle(r) of its row, so that the operand reads
// stay free of bank conflicts: K is read as whole 16-byte chunks, 16 rows per
// access, V by the transposing 8-byte reads, 4 rows x 64 bytes per access (one
// 64-byte group is a whole row at head dim 32, which needs none).
template <int CPR>
__device__ __forceinline__ int tile_swizzle_k(int r) {
  return CPR == 16 ? (r & 15) : CPR == 8 ? ((r >> 1) & 7) : ((r >> 2) & 3);
}
template <int CPR>
__device__ __forceinline__ int tile_swizzle_v(int r) {
  return CPR == 16 ? ((r & 3) << 2) : CPR == 8 ? (((r >> 1) & 1) << 2) : 0;
}

// First row of sequence i's chunk, and the one behind its last.
__device__ __forceinline__ int chunk_begin(const PrefillKP &p, int i) {
  return p.cu_seqlens_q != nullptr ? p.cu_seqlens_q[i] : (int)(i * p.row_pitch);
}
__device__ __forceinline__ int chunk_end(const PrefillKP &p, int i) {
  return p.cu_seqlens_q != nullptr ? p.cu_seqlens_q[i + 1] : (int)(i * p.row_pitch) + p.max_chunk;
}

// The sequence that is `rank`th by context length (longest first: workgroups
// are dispatched in id order and should end together), its first query row,
// context length and chunk length.  Up to one sequence per lane is ranked on
// the fly; in longer batches rank r is simply sequence r.  Equal sequences
// (no context_lens) need no look at memory.
__device__ __forceinline__ void pick_sequence(const PrefillKP &p, int rank, int &seq, int &q_lo, int &L, int &C) {
  seq = rank;
  if (p.context_lens == nullptr) {
    q_lo = (int)(seq * p.row_pitch);
    L = p.uniform_context;
    C = p.max_chunk;
    return;
  }
  const int n_seqs = p.n_units / p.gn;
  if (n_seqs <= kWave) {
    // (the chunk bounds travel with the context lengths, one sequence per lane: the chosen
    // sequence's come from its lane instead of a second round trip to memory)
    const int ln = threadIdx.x & (kWave - 1);
    const int mine = ln < n_seqs ? p.context_lens[ln] : -0x7fffffff;
    const int lo_mine = ln < n_seqs ? chunk_begin(p, ln) : 0;
    const int hi_mine = ln < n_seqs ? chunk_end(p, ln) : 0;
    int above = 0;
    for (int j = 0; j < n_seqs; ++j) {
      const int other = __builtin_amdgcn_readlane(mine, j);
      above += (other > mine || (other == mine && j < ln)) ? 1 : 0;
    }
    const uint64_t hit = __ballot(above == rank && ln < n_seqs);
    seq = __builtin_amdgcn_readfirstlane((int)__builtin_ctzll(hit | (1ull << 63)));
    seq = seq < n_seqs ? seq : n_seqs - 1;
    q_lo = __builtin_amdgcn_readlane(lo_mine, seq);
    L = __builtin_amdgcn_readlane(mine, seq);
    C = __builtin_amdgcn_readlane(hi_mine, seq) - q_lo;
  } else {
    q_lo = chunk_begin(p, seq);
    L = p.context_lens[seq];
    C = chunk_end(p, seq) - q_lo;
  }
}

// Row of q and out that is row r of the chunk whose rows start at q_lo.
__device__ __forceinline__ int64_t query_row(const PrefillKP &p, int q_lo, int r) {
  int64_t row = q_lo + r;
  if (p.rows != nullptr) {
    row = p.rows[row < p.n_rows ? row : p.n_rows - 1];
    row = row < 0 ? 0 : row;  // a corrupt entry must not become an address outside the tensors
    row = row < p.q_rows ? row : p.q_rows - 1;
  }
  return row;
}

// The tiles a query tile visits under a packed mask: entry i (clamped to the last one) holds the tile and the
// classes of the query tile's four 32-row groups.
struct MaskList {
  typedef const __attribute__((address_space(4))) int32_t *ScalarPtr;  // scalar (SMEM) loads
  ScalarPtr at;
  int count;
  const uint64_t *words;  // of the wave's row group: [tile][32]
  __device__ __forceinline__ void open(const PrefillKP &p, int seq, int head, int qtile, int group) {
    const int64_t plane = (int64_t)seq * p.mask_plane_seq + (int64_t)head * p.mask_plane_head;
    at = (ScalarPtr)(unsigned long long)(p.mask_lists + (plane * p.mask_qtiles + qtile) * (p.mask_tiles + 1));
    count = at[0];
    words = p.mask_bits + ((plane * p.mask_qtiles + qtile) * 4 + group) * p.mask_tiles * 32;
  }
  __device__ __forceinline__ int32_t entry(int i) const { return at[1 + (i < count ? i : count - 1)]; }
  static __device__ __forceinline__ int tile(int32_t e) { return e & 0xffff; }
  static __device__ __forceinline__ int kind(int32_t e, int group) { return (e >> (16 + 2 * group)) & 3; }
};

// The rotary tables' row of query row `row` (clamped into them).
__device__ __forceinline__ int rope_position(const PrefillKP &p, int64_t row) {
  int pos = p.positions[row];
  pos = pos < 0 ? 0 : pos;
  return pos >= p.table_rows ? p.table_rows - 1 : pos;
}
__device__ __forceinline__ int64_t rope_row(const PrefillKP &p, int64_t row) {
  return (int64_t)rope_position(p, row) * p.half_hd;
}

constexpr float kLazySlack = 8.0f;  // log2 units

// 16-bit pools, short work: the kernel of paged_prefill_short.hip, and whether a call is that.
bool prefill_takes_short(const PrefillArgs &a);
int launch_paged_prefill_short(PrefillKP kp, const PrefillArgs &a, hipStream_t stream);
// fp32 pools: the kernel of paged_prefill_f32.hip (same parameters, same grid rules of its own).
int launch_paged_prefill_f32(PrefillKP kp, const PrefillArgs &a, hipStream_t stream);

}  // namespace prefill
}  // namespace ic
