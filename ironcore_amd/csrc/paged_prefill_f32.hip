// Chunked prefill against the block KV cache for fp32 pools.
//
// Same contract as the 16-bit kernel of paged_prefill.hip (the reference's
// dense attention, ironcore/layers/attention.py:68-142, with sq = C, sk = L
// and the causal mask of ironcore/language_model.py:109-114 shifted by the
// cached prefix, no mask, or a caller's byte mask), with every product, sum
// and probability in fp32: the dtype the reference's own contract tests feed
// the layer (tests/test_attention.py:143-161).
//
// Flash-attention shape on the fp32 matrix instruction (v_mfma_f32_32x32x2_f32):
//
//  * One workgroup = 128 query rows of one query head: 4 waves, each owning 32
//    rows for the whole K/V sweep.  The wave's query rows stay in registers as
//    MFMA B operands.
//  * K/V are walked in tiles of 32 tokens.  All 256 threads fetch a tile from
//    the pool through the block table (16 bytes per lane and load, rows past
//    the context clamped to the last one) a whole tile ahead, hold it in
//    registers while the current tile is computed, then leave it in the other
//    of two LDS buffers: a K/V byte crosses the memory system once per 128
//    query rows, and there is one workgroup barrier per tile.
//  * S^T = K Q^T: a lane supplies K[token lane % 32][d] and Q[query lane % 32][d]
//    for one d per MFMA; the k index of MFMA 4j + e is d = 8j + 4(lane / 32) + e,
//    so that a lane's four operands of a group are one 16-byte LDS read.  K rows
//    are padded by 4 floats, which spreads the 16 rows of an access over all
//    banks.  A lane then holds one query column of the scores: row maximum and
//    row sum are in-lane reductions plus one exchange between the lane halves.
//  * O^T += V^T P^T: the probabilities are already B operands (MFMA i of a
//    lane half takes the token that half holds in register i), the matching
//    V^T operand is one float per lane from the row-major V tile (rows padded
//    by 8 floats: the two halves read rows 4 apart, on disjoint banks).
//  * Tiles wholly above the causal diagonal are skipped per wave.
//
// FLOPs per launch: 4*hn*hd per visible (query, key) pair, as for the 16-bit
// kernel; bound by the fp32 matrix rate (157 TFLOP/s nominal).
#include "prefill_common.h"
#include "../../include/ironcore_paged.h"

namespace ic {
namespace prefill {

namespace {

constexpr int kF32Waves = 4;
constexpr int kF32Threads = kF32Waves * kWave;
constexpr int kF32BM = kF32Waves * 32;  // query rows per workgroup
constexpr int kF32BN = 32;              // tokens per K/V tile

// MASK: 0 the causal rule or none, 1 a byte mask, 2 a packed one (equal sequences).
template <int HD, bool SINGLE, int MASK>
__global__ __launch_bounds__(kF32Threads) void paged_prefill_f32_kernel(const PrefillKP p) {
  constexpr int NJ = HD / 8;            // 16-byte operand groups of the QK contraction
  constexpr int OB = HD / 32;           // 32-wide blocks of the output head dim
  constexpr int F4R = HD / 4;           // 16-byte pieces per token row
  constexpr int RP = kF32Threads / F4R; // token rows one pass of the workgroup covers
  constexpr int NP = kF32BN / RP;       // passes (pieces per thread and pool) per tile
  constexpr int KP = HD + 4;            // LDS row pitch of K, floats
  constexpr int VP = HD + 8;            // ... of V
  static_assert(HD % 32 == 0 && kF32Threads % F4R == 0 && kF32BN % RP == 0 && NP >= 1, "tile staging shape");

  __shared__ __attribute__((aligned(16))) float s_k[2][kF32BN * KP];
  __shared__ __attribute__((aligned(16))) float s_v[2][kF32BN * VP];

  const int seq = blockIdx.y;
  const int h = blockIdx.x / p.n_qtiles;
  const int q0 = (p.n_qtiles - 1 - blockIdx.x % p.n_qtiles) * kF32BM;  // last query tiles (the longest) first
  const int kvh = h / p.group;
  const bool equal = p.context_lens == nullptr;  // equal sequences: nothing to look up
  const int q_lo = chunk_begin(p, seq);
  int L = equal ? p.uniform_context : p.context_lens[seq];
  int C = chunk_end(p, seq) - q_lo;
  const bool causal = MASK == 0 && p.causal;
  if (L < 0) L = 0;
  if (causal && C > L) C = L;  // under the causal rule a chunk cannot be longer than its context
  if (q0 >= C) return;
  const int tid = threadIdx.x;
  if (L == 0) {  // query rows without any key (not under the causal rule): zero rows
    const int rows = C - q0 < kF32BM ? C - q0 : kF32BM;
    for (int idx = tid; idx < rows * F4R; idx += kF32Threads)
      store16(p.out + (query_row(p, q_lo, q0 + idx / F4R) * p.out_stride_token + (int64_t)h * HD + (idx % F4R) * 4) * 4,
              Vec16{{0u, 0u, 0u, 0u}});
    return;
  }
  const int P = L - C;  // cached prefix (causal rule only)
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int n = lane & 31;   // query column of this lane within the wave's 32-row block
  const int hh = lane >> 5;  // which operand of each k pair this lane feeds

  // ---- query rows: registers for the whole sweep, as MFMA B operands ------------
  const int my_q = q0 + wave * 32 + n;
  const int qrow = my_q < C ? my_q : C - 1;
  const int limit = causal ? P + qrow : L - 1;  // last key this query row may see
  const int64_t at_row = query_row(p, q_lo, qrow);
  float4 qf[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    qf[j] = *reinterpret_cast<const float4 *>(
        p.q + (at_row * p.q_stride_token + (int64_t)h * HD + 8 * j + 4 * hh) * 4);
  if (p.positions != nullptr) {
    const int64_t trig = rope_row(p, at_row) + 2 * hh;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      qf[j] = __builtin_bit_cast(float4, rotate_chunk<F32>(__builtin_bit_cast(Vec16, qf[j]), p.cos_table + trig + 4 * j,
                                                           p.sin_table + trig + 4 * j));
  }

  f32x16_t o[OB];
  float m = kNegInf, l = 0.f;
#pragma unroll
  for (int ob = 0; ob < OB; ++ob)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[ob][i] = 0.f;

  int kv_end = causal ? P + q0 + kF32BM : L;  // keys any row of this workgroup can see
  kv_end = kv_end < L ? kv_end : L;
  // (a packed mask's list is of 64-key tiles: two tiles of this kernel each)
  MaskList list;
  if constexpr (MASK == 2) list.open(p, seq, h, q0 / kF32BM, wave);
  const int n_tiles = MASK == 2 ? 2 * list.count : (kv_end + kF32BN - 1) / kF32BN;
  int my_end = causal ? P + q0 + wave * 32 + 32 : L;
  my_end = my_end < kv_end ? my_end : kv_end;
  const int my_tiles = (my_end > 0 && q0 + wave * 32 < C) ? (my_end + kF32BN - 1) / kF32BN : 0;

  // ---- tile staging: memory -> registers (a tile ahead) -> LDS -------------------------
  const int r0 = tid / F4R;  // first token row of the tile this thread fetches
  const int c4 = tid % F4R;  // its 16-byte piece of the row
  const int32_t *table_row = p.block_tables + (int64_t)seq * p.bt_stride;
  const int64_t head_off = (int64_t)kvh * p.stride_head + c4 * 4;
  // tile t of the sweep: its number, and under a packed mask the class of this wave's rows and the words
  auto number = [&](int t) { return MASK == 2 ? 2 * MaskList::tile(list.entry(t >> 1)) + (t & 1) : t; };
  uint32_t word = 0, word_next = 0;  // packed mask: this lane's row, tile t and t + 1
  auto fetch = [&](int t, Vec16 *kr, Vec16 *vr) {
    const int tile = number(t);
    if constexpr (MASK == 2) word_next = reinterpret_cast<const uint32_t *>(list.words)[((tile >> 1) * 32 + n) * 2 + (tile & 1)];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      int tok = tile * kF32BN + r0 + i * RP;
      tok = tok < L ? tok : L - 1;  // rows past the context: a valid row, never visible
      int blk = 0, within = tok;
      if (!SINGLE) {
        blk = p.block_shift >= 0 ? tok >> p.block_shift : tok / p.block_size;
        within = tok - blk * p.block_size;
      }
      int64_t phys = SINGLE && p.block_tables == nullptr ? seq : table_row[blk];
      // A corrupt table entry must not become an out-of-pool address.
      phys = phys < 0 ? 0 : phys;
      phys = phys >= p.num_blocks ? p.num_blocks - 1 : phys;
      const int64_t off = (phys * p.stride_block + head_off + (int64_t)within * p.stride_token) * 4;
      kr[i] = load16(p.k_pool + off);
      vr[i] = load16(p.v_pool + off);
    }
  };
  auto stash = [&](int buf, const Vec16 *kr, const Vec16 *vr) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      store16(&s_k[buf][(r0 + i * RP) * KP + c4 * 4], kr[i]);
      store16(&s_v[buf][(r0 + i * RP) * VP + c4 * 4], vr[i]);
    }
  };

  f32x16_t s;  // S^T of the tile: (token, query n); after the softmax its probabilities

  // ---- S^T = K Q^T ----------------------------------------------------------------
  auto scores = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    const float *kb = &s_k[buf][n * KP + 4 * hh];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float4 a = *reinterpret_cast<const float4 *>(kb + 8 * j);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, qf[j].x, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, qf[j].y, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, qf[j].z, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, qf[j].w, s, 0, 0, 0);
    }
  };
  // ---- softmax of the tile's scores: s -> probabilities, m, l (and o when the reference moves) ----
  auto softmax = [&](int tile, int kind) {
    // s[i] is (token tile*32 + 4*hh + 8*(i/4) + i%4, query n)
    const int tok_base = tile * kF32BN + 4 * hh;
    const bool need_mask = causal ? (tile * kF32BN + kF32BN - 1 > P + q0 + wave * 32) : (tile * kF32BN + kF32BN > L);
    if (need_mask) {  // tiles that touch the causal diagonal (or the context end)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int tok = tok_base + 8 * (i / 4) + (i & 3);
        s[i] = tok > limit ? kNegInf : s[i];
      }
    }
    if constexpr (MASK == 1) {  // keys the caller's mask hides from this lane's query row
      const uint8_t *mrow = p.mask + (int64_t)seq * p.mask_stride_seq + (int64_t)h * p.mask_stride_head +
                            (int64_t)qrow * p.mask_stride_row;
      // unconditional loads from an index clamped into the part of the row that exists and counts
      const int last = (limit < p.mask_keys - 1 ? limit : p.mask_keys - 1);
      uint8_t seen[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int tok = tok_base + 8 * (i / 4) + (i & 3);
        seen[i] = mrow[tok < last ? tok : last];
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int tok = tok_base + 8 * (i / 4) + (i & 3);
        const bool hidden = (tok <= limit) & ((tok >= p.mask_keys) | (seen[i] == 0));
        s[i] = hidden ? kHiddenScore : s[i];
      }
    }
    if (MASK == 2 && kind == 1) {
      const uint32_t w = word >> (4 * hh);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const bool hidden = (w & (1u << (8 * (i / 4) + (i & 3)))) == 0;
        s[i] = hidden ? fminf(s[i], kHiddenScore) : s[i];
      }
    }
    float mx = kNegInf;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
    float mx_a, mx_b;
    both_halves(mx, mx_a, mx_b);
    mx = fmaxf(mx_a, mx_b) * p.scale_log2e;
    // Lazy reference maximum, as in the 16-bit kernel: it moves (and the accumulators are
    // rescaled) only when some row's maximum rises more than 2^kLazySlack above it.
    if (__any(mx > m + kLazySlack)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = (m == kNegInf) ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int ob = 0; ob < OB; ++ob)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[ob][i] *= alpha;
    }
    const float neg_ms = (m == kNegInf) ? 0.f : -m;
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], p.scale_log2e, neg_ms));
      ps += s[i];
    }
    l += ps;
  };
  // ---- O^T += V^T P^T ---------------------------------------------------------------
  auto weighted_values = [&](int buf) {
    const float *vb = &s_v[buf][4 * hh * VP + n];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float *row = vb + ((i & 3) + 8 * (i >> 2)) * VP;  // token (i%4) + 8(i/4) + 4hh of the tile
#pragma unroll
      for (int ob = 0; ob < OB; ++ob) o[ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(row[ob * 32], s[i], o[ob], 0, 0, 0);
    }
  };

  Vec16 kr[NP], vr[NP];
  fetch(0, kr, vr);
  stash(0, kr, vr);
  __syncthreads();
  for (int t = 0; t < n_tiles; ++t) {
    const bool more = t + 1 < n_tiles;  // the same for every wave of the workgroup
    word = word_next;
    if (more) fetch(t + 1, kr, vr);
    const int tile = number(t);
    const int kind = MASK == 2 ? MaskList::kind(list.entry(t >> 1), wave) : 2;
    // (the second half of a packed mask's last tile may lie past the context altogether)
    if (MASK == 2 ? (kind != 0 && tile * kF32BN < L && q0 + wave * 32 < C) : t < my_tiles) {
      scores(t & 1);
      softmax(tile, kind);
      weighted_values(t & 1);
    }
    // buffer (t + 1) & 1 was last read for tile t - 1, before the barrier that ended that round
    if (more) stash((t + 1) & 1, kr, vr);
    __syncthreads();
  }

  // ---- normalise and store -------------------------------------------------------
  float l_a, l_b;
  both_halves(l, l_a, l_b);
  const float lt = l_a + l_b;
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  if (my_q < C) {
    float *orow = reinterpret_cast<float *>(p.out) + query_row(p, q_lo, my_q) * p.out_stride_token + (int64_t)h * HD;
#pragma unroll
    for (int ob = 0; ob < OB; ++ob) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = ob * 32 + 4 * hh + 8 * j;
        *reinterpret_cast<float4 *>(orow + d) = make_float4(o[ob][4 * j] * inv, o[ob][4 * j + 1] * inv,
                                                            o[ob][4 * j + 2] * inv, o[ob][4 * j + 3] * inv);
      }
    }
  }
}

// The same for grids that leave the GPU idle.  The kernel above gives a workgroup 128 rows and a wave a serial sweep of its
// 32 rows over all keys, 3.9 us a tile at head dim 128 (128 matrix instructions of 64 cycles), whether or not there are
// other rows to share the tiles with: a chunk of 30 rows keeps one wave of a CU busy.  Here a workgroup has 32 rows and its
// four waves take the tiles in turn, each with its own sums, merged through LDS at the end.  (When: takes_split.)  A wave reads its tiles
// straight into matrix operands: K 16 bytes a lane of the lane's token, V a word a lane of 32 neighbours; K of the next
// tile is asked for when the scores are done and arrives under the weighted values, V the other way round, so there is
// neither staging nor a barrier.  One wave to a SIMD (some 300 registers).  Bound by the matrix instructions of a
// wave's share, with one round trip at either end.
template <int HD, bool SINGLE>
__global__ __launch_bounds__(kF32Threads) void paged_prefill_f32_split_kernel(const PrefillKP p) {
  constexpr int NJ = HD / 8;
  constexpr int OB = HD / 32;
  constexpr int F4R = HD / 4;
  __shared__ __attribute__((aligned(16))) float s_o[kF32Waves][OB * 16][kWave];
  __shared__ float s_m[kF32Waves][32], s_l[kF32Waves][32];

  const int seq = blockIdx.y;
  const int h = blockIdx.x / p.n_qtiles;
  const int q0 = (p.n_qtiles - 1 - blockIdx.x % p.n_qtiles) * 32;  // the longest first
  const int kvh = h / p.group;
  const bool equal = p.context_lens == nullptr;
  const int q_lo = chunk_begin(p, seq);
  int L = equal ? p.uniform_context : p.context_lens[seq];
  int C = chunk_end(p, seq) - q_lo;
  const bool causal = p.causal;
  if (L < 0) L = 0;
  if (causal && C > L) C = L;
  if (q0 >= C) return;
  const int tid = threadIdx.x;
  if (L == 0) {
    const int rows = C - q0 < 32 ? C - q0 : 32;
    for (int idx = tid; idx < rows * F4R; idx += kF32Threads)
      store16(p.out + (query_row(p, q_lo, q0 + idx / F4R) * p.out_stride_token + (int64_t)h * HD + (idx % F4R) * 4) * 4,
              Vec16{{0u, 0u, 0u, 0u}});
    return;
  }
  const int P = L - C;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int n = lane & 31, hh = lane >> 5;
  const int my_q = q0 + n;
  const int qrow = my_q < C ? my_q : C - 1;
  const int limit = causal ? P + qrow : L - 1;
  const int64_t at_row = query_row(p, q_lo, qrow);

  int kv_end = causal ? P + q0 + 32 : L;
  kv_end = kv_end < L ? kv_end : L;
  const int n_tiles = (kv_end + kF32BN - 1) / kF32BN;
  const int32_t *table_row = p.block_tables + (int64_t)seq * p.bt_stride;
  // byte offset of a tile's token n in the pools (rows past the context: the last one, never visible)
  auto token_row = [&](int t) {
    int tok = (t < n_tiles ? t : 0) * kF32BN + n;
    tok = tok < L ? tok : L - 1;
    int blk = 0, within = tok;
    if (!SINGLE) {
      blk = p.block_shift >= 0 ? tok >> p.block_shift : tok / p.block_size;
      within = tok - blk * p.block_size;
    }
    int64_t phys = SINGLE && p.block_tables == nullptr ? seq : table_row[blk];
    phys = phys < 0 ? 0 : phys;  // a corrupt table entry must not become an out-of-pool address
    phys = phys >= p.num_blocks ? p.num_blocks - 1 : phys;
    return (phys * p.stride_block + (int64_t)kvh * p.stride_head + (int64_t)within * p.stride_token) * 4;
  };
  float4 kf[NJ];
  float vf[16][OB];
  auto fetch_k = [&](int64_t row) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) kf[j] = *reinterpret_cast<const float4 *>(p.k_pool + row + 32 * j + 16 * hh);
  };
  // Matrix instruction i takes token (i % 4) + 8 (i / 4) of a tile in one half of the lanes and the fourth after it in the
  // other.  Eight tokens lie at one stride where they are all there and in one block; else each lane asks the lane that
  // has the token's row.
  const bool strided = (SINGLE || p.block_size % 8 == 0) && p.stride_token < 1 << 24;
  const uint32_t pitch = (uint32_t)p.stride_token * 4, in_group = (4 * hh) * pitch + n * 4;
  auto fetch_v = [&](int t, int64_t row) {
    const uint32_t lo = (uint32_t)row, hi = (uint32_t)((uint64_t)row >> 32);
    if (strided && (t + 1) * kF32BN <= L) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t first = (int64_t)(((uint64_t)__builtin_amdgcn_readlane(hi, 8 * q) << 32) |
                                        (uint32_t)__builtin_amdgcn_readlane(lo, 8 * q));
        const char *base = p.v_pool + first;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int ob = 0; ob < OB; ++ob)
            vf[4 * q + i][ob] = *reinterpret_cast<const float *>(base + (in_group + i * pitch) + ob * 128);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int from = (i & 3) + 8 * (i >> 2) + 4 * hh;
      const char *at = p.v_pool + (int64_t)(((uint64_t)(uint32_t)__shfl(hi, from, kWave) << 32) | (uint32_t)__shfl(lo, from, kWave)) + n * 4;
#pragma unroll
      for (int ob = 0; ob < OB; ++ob) vf[i][ob] = *reinterpret_cast<const float *>(at + ob * 128);
    }
  };
  int t = wave;
  int64_t row = token_row(t), row_next = 0;
  fetch_k(row);
  fetch_v(t < n_tiles ? t : 0, row);
  float4 qf[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    qf[j] = *reinterpret_cast<const float4 *>(p.q + (at_row * p.q_stride_token + (int64_t)h * HD + 8 * j + 4 * hh) * 4);
  if (p.positions != nullptr) {
    const int64_t trig = rope_row(p, at_row) + 2 * hh;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      qf[j] = __builtin_bit_cast(float4, rotate_chunk<F32>(__builtin_bit_cast(Vec16, qf[j]), p.cos_table + trig + 4 * j,
                                                           p.sin_table + trig + 4 * j));
  }
  f32x16_t o[OB];
  float m = kNegInf, l = 0.f;
#pragma unroll
  for (int ob = 0; ob < OB; ++ob)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[ob][i] = 0.f;
  while (t < n_tiles) {
    const int after = t + kF32Waves;
    if (after < n_tiles) row_next = token_row(after);
    // two sums, since an instruction that adds to the last one's result waits for it
    f32x16_t s, s2;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = s2[i] = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j].x, qf[j].x, s, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j].y, qf[j].y, s2, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j].z, qf[j].z, s, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j].w, qf[j].w, s2, 0, 0, 0);
    }
    if (after < n_tiles) fetch_k(row_next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] += s2[i];
    const int tok_base = t * kF32BN + 4 * hh;
    if (causal ? (t * kF32BN + kF32BN - 1 > P + q0) : (t * kF32BN + kF32BN > L)) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = tok_base + 8 * (i / 4) + (i & 3) > limit ? kNegInf : s[i];
    }
    float mx = kNegInf;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
    float mx_a, mx_b;
    both_halves(mx, mx_a, mx_b);
    mx = fmaxf(mx_a, mx_b) * p.scale_log2e;
    if (__any(mx > m + kLazySlack)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = (m == kNegInf) ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int ob = 0; ob < OB; ++ob)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[ob][i] *= alpha;
    }
    const float neg_ms = (m == kNegInf) ? 0.f : -m;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], p.scale_log2e, neg_ms));
      l += s[i];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int ob = 0; ob < OB; ++ob) o[ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[i][ob], s[i], o[ob], 0, 0, 0);
    if (after < n_tiles) fetch_v(after, row_next);
    __builtin_amdgcn_sched_barrier(0);
    t = after;
  }
  // ---- merge -------------------------------------------------------------------------
  float l_a, l_b;
  both_halves(l, l_a, l_b);
  if (hh == 0) s_m[wave][n] = m, s_l[wave][n] = l_a + l_b;
#pragma unroll
  for (int ob = 0; ob < OB; ++ob)
#pragma unroll
    for (int i = 0; i < 16; ++i) s_o[wave][ob * 16 + i][lane] = o[ob][i];
  __syncthreads();
  float top = kNegInf, lt = 0.f, weight[kF32Waves];
#pragma unroll
  for (int w = 0; w < kF32Waves; ++w) top = fmaxf(top, s_m[w][n]);
#pragma unroll
  for (int w = 0; w < kF32Waves; ++w) {
    weight[w] = s_m[w][n] == kNegInf ? 0.f : __builtin_amdgcn_exp2f(s_m[w][n] - top);
    lt = __builtin_fmaf(s_l[w][n], weight[w], lt);
  }
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  if (my_q >= C) return;
  float *orow = reinterpret_cast<float *>(p.out) + query_row(p, q_lo, my_q) * p.out_stride_token + (int64_t)h * HD;
#pragma unroll
  for (int ob = 0; ob < OB; ++ob) {  // four dims of each block to a wave
    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) {
      const int at = ob * 16 + 4 * wave;
      sum.x = __builtin_fmaf(s_o[w][at][lane], weight[w], sum.x), sum.y = __builtin_fmaf(s_o[w][at + 1][lane], weight[w], sum.y);
      sum.z = __builtin_fmaf(s_o[w][at + 2][lane], weight[w], sum.z), sum.w = __builtin_fmaf(s_o[w][at + 3][lane], weight[w], sum.w);
    }
    *reinterpret_cast<float4 *>(orow + ob * 32 + 4 * hh + 8 * wave) = make_float4(sum.x * inv, sum.y * inv, sum.z * inv, sum.w * inv);
  }
}

template <bool SINGLE>
int launch_split(const PrefillKP &kp, int hd, dim3 grid, hipStream_t stream) {
  switch (hd) {
    case 32:
      hipLaunchKernelGGL((paged_prefill_f32_split_kernel<32, SINGLE>), grid, dim3(kF32Threads), 0, stream, kp);
      break;
    case 64:
      hipLaunchKernelGGL((paged_prefill_f32_split_kernel<64, SINGLE>), grid, dim3(kF32Threads), 0, stream, kp);
      break;
    case 128:
      hipLaunchKernelGGL((paged_prefill_f32_split_kernel<128, SINGLE>), grid, dim3(kF32Threads), 0, stream, kp);
      break;
    default:
      return IC_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

template <bool SINGLE, int MASK>
int launch_hd(const PrefillKP &kp, int hd, dim3 grid, hipStream_t stream) {
  switch (hd) {
    case 32:
      hipLaunchKernelGGL((paged_prefill_f32_kernel<32, SINGLE, MASK>), grid, dim3(kF32Threads), 0, stream, kp);
      break;
    case 64:
      hipLaunchKernelGGL((paged_prefill_f32_kernel<64, SINGLE, MASK>), grid, dim3(kF32Threads), 0, stream, kp);
      break;
    case 128:
      hipLaunchKernelGGL((paged_prefill_f32_kernel<128, SINGLE, MASK>), grid, dim3(kF32Threads), 0, stream, kp);
      break;
    default:
      return IC_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

// Whether the rows are cut finer and the keys split.  us of 128 rows to a workgroup / of 32, by blocks of 32 rows (chunks and
// heads together) and 32-key tiles of the longest sweep:
//   hd 128, 1 chunk of 100 behind 4 000, 32 heads        128 blocks, 129 tiles   353 / 89
//           3 of 172-284 behind up to 74, 8              216         12           56 / 24
//           4 of 4-261 behind up to 275, 16              576         17           80 / 49
//           21 of 69 behind up to 1 587, 12              756         52          291 / 178
//           4 of 1 264, 8, dense                       1 280         40          271 / 182
//           2 of 806 behind up to 56, 32               1 664         27          216 / 188
//           4 of 600, 32                               2 432         19          238 / 232
//           1 of 2 000, 8, dense without a mask          504         63          285 / 150
//           36 of 73, 8, dense                           864          3         32.5 / 37.1
//           50 of 25, 32, dense                        1 600          1         33.8 / 58.0
//   hd 64   2 of 75, 32, dense                           192          3         10.9 / 8.8
//           7 of 437, 8                                  784         14         48.8 / 43.0
//           8 of 300, 12                                 960         10         55.5 / 43.1
//           20 of 129, 12, dense                       1 200          5         24.6 / 26.6
//           8 of 500, 16, dense without a mask         2 048         16         76.7 / 98.8
//           12 of 117 behind up to 899, 64             3 072         32          165 / 172
// and the sweeps of few tiles (paged but for the dense ones):
//   hd 128  16 of 73, 16                               768          3         32.4 / 40.2
//           9 of 40, 16, dense                         288          2         13.4 / 19.6
//           15 of 129, 8, dense                        600          5         27.1 / 36.2
//           14 of 200, 8                               784          7         54.7 / 56.7
//           25 of 40 behind 150, 16                    800          6         80.6 / 73.4
//           15 of 129 behind 140, 8                    600          9         67.3 / 63.3
//           38 of 20 behind 250, 16                    608          9          160 / 70
//   hd 64   16 of 73, 16                               768          3         20.6 / 25.3
//           14 of 200, 8, dense                        784          7         21.9 / 25.5
//           8 of 280, 8, dense                         576          9         25.9 / 23.1
//           13 of 64 behind 210, 16                    416          9         36.3 / 27.0
// Long sweeps split until the matrix units are busy either way, later under the causal rule over long chunks, whose
// workgroups are of unequal length; short ones only while each block has a CU to itself.  (The tables' width stands for the
// longest context only where the caller does not say it: a table may have room for many more blocks.)
bool takes_split(const PrefillArgs &a) {
  if (a.mask != nullptr || a.mask_bits != nullptr) return false;
  const bool one_block = a.block_tables == nullptr || a.block_table_stride == 1;
  if (!one_block && a.pool.block_size < 1) return false;
  const int64_t blocks = ((int64_t)a.max_chunk_len + 31) / 32 * a.hn * a.n_seqs;
  const int64_t cus = device_cu_count();
  int64_t keys = a.uniform_context;
  if (a.context_lens != nullptr) {
    const int64_t width = a.block_table_stride * a.pool.block_size;
    keys = keys > 0 && keys < width ? keys : width;
  }
  if (keys <= 7 * kF32BN) return blocks <= cus;
  return blocks <= (a.causal && a.max_chunk_len >= 300 ? 53 : 25) * cus / 8;
}

}  // namespace

int launch_paged_prefill_f32(PrefillKP kp, const PrefillArgs &a, hipStream_t stream) {
  kp.n_qtiles = (a.max_chunk_len + kF32BM - 1) / kF32BM;
  const int64_t wgs_x = (int64_t)kp.n_qtiles * a.hn;
  if (wgs_x > 0x7fffffff || a.n_seqs > 65535) return IC_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)wgs_x, (unsigned)a.n_seqs);
  const bool masked = a.mask != nullptr;
  if (takes_split(a)) {
    kp.n_qtiles = (a.max_chunk_len + 31) / 32;
    const dim3 fine((unsigned)(kp.n_qtiles * a.hn), (unsigned)a.n_seqs);
    return a.block_tables == nullptr || a.block_table_stride == 1 ? launch_split<true>(kp, a.hd, fine, stream)
                                                                  : launch_split<false>(kp, a.hd, fine, stream);
  }
  if (a.mask_bits != nullptr) return launch_hd<true, 2>(kp, a.hd, grid, stream);
  // A one-column block table means one block per sequence, of any length.
  if (a.block_tables == nullptr || a.block_table_stride == 1)
    return masked ? launch_hd<true, 1>(kp, a.hd, grid, stream) : launch_hd<true, 0>(kp, a.hd, grid, stream);
  if (kp.block_size < 1) return IC_ERR_UNSUPPORTED;
  return masked ? launch_hd<false, 1>(kp, a.hd, grid, stream) : launch_hd<false, 0>(kp, a.hd, grid, stream);
}

}  // namespace prefill
}  // namespace ic
