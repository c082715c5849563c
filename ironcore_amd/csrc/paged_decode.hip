// Paged decode: one query token per sequence against the block KV cache.
//
// What it computes is the reference's dense attention with sq = 1
// (ironcore/layers/attention.py:68-142) on the rows the block table names:
// scores = q.k * scale, softmax over the context, out = probs @ v, with query
// head h reading KV head h / G (attention.py:95-102).
//
// This file holds the host-side launch, the split-K reduce pass and the
// vector-ALU main kernel, which is the one fp32 pools run on (scores, softmax
// and the PV sum stay in fp32).  bf16 and fp16 pools take the matrix-core main
// kernel of paged_decode_mfma.hip; both share everything described here
// except the arithmetic of a tile.
//
// HBM-bound streaming kernel (one pass over every visible K and V byte).
//
//  * Unit of work: a TILE = 16 consecutive tokens of one (sequence, KV head)
//    "pair" (one pool block at block size 16, a slice of a longer block
//    otherwise), for ALL G query heads that share the KV head, so each K/V
//    byte is fetched once per KV head, not once per query head.  (G > 8 is
//    cut into sub-groups of <= 8 heads, each its own pair.)
//  * Split-K by equal shares: the tiles of the whole batch form one sequence
//    (pair-major, block-minor); every resident WAVE prefix-sums the
//    per-sequence block counts and takes one contiguous chunk of
//    ceil(N / waves) tiles.  A chunk may start and end inside a pair and may
//    span several pairs; each (wave, pair) segment yields one partial.  All
//    waves carry the same load whatever the spread of context lengths, the
//    grid is exactly the number of waves the GPU holds at once, and waves
//    never synchronise with each other.  Shares are dealt XCD-major, so
//    neighbouring shares (which may alias the same prefix blocks) share an L2.
//  * At the start of its chunk a wave gathers the byte offsets of its next
//    256 tiles from the block table, one per lane and slot; the loop reads
//    them back as wave-uniform scalars (v_readlane), so the table is off the
//    load path and tile addresses are SALU work.
//  * One tile is block_size*hd contiguous elements per K and per V; each lane
//    fetches 16 bytes per load, so one load instruction covers 1 KiB of
//    consecutive bytes (64/LPR token rows, LPR = lanes per row).  Two
//    register tiles in ping-pong: the next tile's loads are in flight while
//    the current one is consumed, across pair boundaries too; the next
//    pair's query is prefetched a segment ahead.
//  * q.k: fused multiply-adds (v_dot2 for 16-bit types), then a DPP butterfly
//    over the LPR lanes that share a row.  Online softmax per lane group; p*v
//    accumulates into EPL fp32 registers per query head with no cross-lane
//    traffic.
//  * Segment end: the lane groups of the wave are merged (log-sum-exp) through
//    a private LDS slab.  A segment that covers its whole pair writes the
//    output row; otherwise (m, l, acc) go to the workspace and the reduce
//    kernel combines the few partials of that pair.
//
// Algorithmic bytes per launch: sum_i ctx_i * 2 * gn * hd * elem (K and V,
// once per KV head) + q, out, block-table entries and context lengths.
#include "decode_common.h"
#include "decode_pair.h"
#include "rope_device.h"
#include "../../include/ironcore_paged.h"

namespace ic {

using namespace decode;

namespace {

template <class E, int HD, int GT, int BS, int NW>
__global__ __launch_bounds__(NW *kWave) void paged_decode_kernel(const DecodeKP p) {
  using T = typename E::type;
  constexpr int EPL = E::EPL;
  constexpr int ES = sizeof(T);
  constexpr int LPR = HD / EPL;     // lanes sharing one token row
  constexpr int RPL = kWave / LPR;  // token rows per load instruction
  constexpr int NLD = BS / RPL;     // load instructions per tile
  constexpr int SW = 4;             // tile offsets held per lane: a window is 64*SW tiles
  static_assert(HD % EPL == 0 && kWave % LPR == 0 && BS % RPL == 0, "tile shape");

  __shared__ __attribute__((aligned(16))) float s_acc[NW][RPL][GT][HD];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int col = lane % LPR;
  const int rowg = lane / LPR;

  // ---- this wave's share of the batch-wide tile sequence ----------------------
  const int64_t wid = (int64_t)xcd_major_workgroup() * NW + wave;
  int64_t left;  // tiles not yet consumed
  TileCursor c;
  if (!locate_chunk<BS>(p, lane, 0, wid, left, c)) return;
  TileCursor walk = c;  // gathers tile addresses ahead of the arithmetic
  TileCursor peek = c;  // the segment after the current one (its q is prefetched)
  next_pair(p, GlobalRows<BS>{p, 0}, peek);
  int seg_blk0 = c.blk;

  uint32_t lane_off[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i)
    lane_off[i] = (uint32_t)(((i * RPL + rowg) * p.stride_token + col * EPL) * ES);

  auto load_q = [&](const TileCursor &tc, Vec16 *qq) {
    const int kvh = tc.pair / p.nsub;
    const int sub = tc.pair - kvh * p.nsub;
    const int head0 = kvh * p.group + sub * GT;
    const int heads = (p.group - sub * GT < GT) ? p.group - sub * GT : GT;
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      qq[g] = Vec16{{0u, 0u, 0u, 0u}};
      if (g < heads && tc.seq < p.n_seqs)
        qq[g] = load16(p.q + (tc.seq * p.q_stride_seq + (int64_t)(head0 + g) * HD + col * EPL) * ES);
    }
  };
  Vec16 qreg[GT], qnext[GT];
  load_q(c, qreg);
  load_q(peek, qnext);

  float m[GT], l[GT], acc[GT][EPL];
#pragma unroll
  for (int g = 0; g < GT; ++g) {
    m[g] = kNegInf;
    l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[g][e] = 0.f;
  }

  // End of a segment: merge the RPL row groups of the wave (log-sum-exp)
  // through the wave's LDS slab, write the output row or a partial, then move
  // to the next pair.  The next tile's loads are already in flight.
  auto finish_segment = [&]() {
    const int kvh = c.pair / p.nsub;
    const int sub = c.pair - kvh * p.nsub;
    const int head0 = kvh * p.group + sub * GT;
    const int heads = (p.group - sub * GT < GT) ? p.group - sub * GT : GT;
    float lsum[GT], mall[GT];
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      float mx = m[g];
      if (RPL >= 2) mx = fmaxf(mx, __shfl_xor(mx, LPR, kWave));
      if (RPL >= 4) mx = fmaxf(mx, __shfl_xor(mx, 2 * LPR, kWave));
      if (RPL >= 8) mx = fmaxf(mx, __shfl_xor(mx, 4 * LPR, kWave));
      const float w = (m[g] == kNegInf) ? 0.f : __builtin_amdgcn_exp2f(m[g] - mx);
      float ls = l[g] * w;
      if (RPL >= 2) ls += __shfl_xor(ls, LPR, kWave);
      if (RPL >= 4) ls += __shfl_xor(ls, 2 * LPR, kWave);
      if (RPL >= 8) ls += __shfl_xor(ls, 4 * LPR, kWave);
      lsum[g] = ls;
      mall[g] = mx;
#pragma unroll
      for (int e = 0; e < EPL; e += 4) {
        float4 v4 = make_float4(acc[g][e] * w, acc[g][e + 1] * w, acc[g][e + 2] * w, acc[g][e + 3] * w);
        *reinterpret_cast<float4 *>(&s_acc[wave][rowg][g][col * EPL + e]) = v4;
      }
      m[g] = kNegInf;
      l[g] = 0.f;
#pragma unroll
      for (int e = 0; e < EPL; ++e) acc[g][e] = 0.f;
    }
    // Only this wave reads what it wrote: a wave-level fence is enough.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const bool whole_pair = (seg_blk0 == 0 && c.blk == c.nb);
    const int64_t partial = wid + (int64_t)c.seq * p.pairs_per_seq + c.pair;
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      if (g >= heads) break;
      const int h = head0 + g;
#pragma unroll
      for (int d = lane; d < HD; d += kWave) {
        float a = 0.f;
#pragma unroll
        for (int r = 0; r < RPL; ++r) a += s_acc[wave][r][g][d];
        if (whole_pair)
          reinterpret_cast<T *>(p.out)[c.seq * p.out_stride_seq + (int64_t)h * HD + d] =
              E::narrow(a / lsum[g]);
        else
          p.part_acc[(partial * GT + g) * HD + d] = a;
      }
      if (!whole_pair && lane == 0) {
        p.part_ml[(partial * GT + g) * 2] = mall[g];
        p.part_ml[(partial * GT + g) * 2 + 1] = lsum[g];
      }
    }
    // The slab is reused by the next segment.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (left > 0) {
      c = peek;
      seg_blk0 = 0;
#pragma unroll
      for (int g = 0; g < GT; ++g) qreg[g] = qnext[g];
      next_pair(p, GlobalRows<BS>{p, 0}, peek);
      load_q(peek, qnext);
    }
  };

  // One tile of arithmetic on the registers (kk, vv), for the tile at cursor c.
  auto consume = [&](Vec16 *kk, Vec16 *vv) {
    float s[GT][NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
#pragma unroll
      for (int g = 0; g < GT; ++g) {
        float d = E::dot(kk[i], qreg[g], 0.f);
        s[g][i] = group_sum<LPR>(d) * p.scale_log2e;
      }
    }
    if (c.blk == c.nb - 1) {  // the sequence's last block may be partly filled
      int ctx = p.context_lens[c.seq];
      ctx = ctx < p.max_ctx ? ctx : p.max_ctx;
      const int tok0 = c.blk * BS;
      if (tok0 + BS > ctx) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
          if (tok0 + i * RPL + rowg >= ctx) {
#pragma unroll
            for (int g = 0; g < GT; ++g) s[g][i] = kNegInf;
            vv[i] = Vec16{{0u, 0u, 0u, 0u}};
          }
        }
      }
    }
    if (p.key_mask != nullptr) {  // keys the caller's mask hides (context-length cuts stay -inf)
      int ctx = p.context_lens[c.seq];
      ctx = ctx < p.max_ctx ? ctx : p.max_ctx;
      const int kvh = c.pair / p.nsub;
      const int head0 = kvh * p.group + (c.pair - kvh * p.nsub) * GT;
      const uint8_t *mrow = p.key_mask + c.seq * p.key_mask_stride_seq + c.blk * BS + rowg;
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        if (c.blk * BS + i * RPL + rowg < ctx) {
#pragma unroll
          for (int g = 0; g < GT; ++g) {
            const int h = head0 + g < p.hn ? head0 + g : p.hn - 1;
            if (mrow[h * p.key_mask_stride_head + i * RPL] == 0) s[g][i] = kHiddenLog2;
          }
        }
      }
    }
    float vf[NLD][EPL];
#pragma unroll
    for (int i = 0; i < NLD; ++i) E::widen(vv[i], vf[i]);
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      float mx = m[g];
#pragma unroll
      for (int i = 0; i < NLD; ++i) mx = fmaxf(mx, s[g][i]);
      const float ms = (mx == kNegInf) ? 0.f : mx;
      const float alpha = __builtin_amdgcn_exp2f(m[g] - ms);
      float pr[NLD];
      float ps = 0.f;
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        pr[i] = __builtin_amdgcn_exp2f(s[g][i] - ms);
        ps += pr[i];
      }
      l[g] = l[g] * alpha + ps;
      m[g] = mx;
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        float a = acc[g][e] * alpha;
#pragma unroll
        for (int i = 0; i < NLD; ++i) a = __builtin_fmaf(pr[i], vf[i][e], a);
        acc[g][e] = a;
      }
    }
    ++c.blk;
    --left;
    if (c.blk == c.nb || left == 0) finish_segment();
  };

  while (left > 0) {
    // ---- window: byte offsets of the next n_win tiles, one per lane and slot ---
    const int n_win = left < kWave * SW ? (int)left : kWave * SW;
    uint32_t off_lo[SW], off_hi[SW];
    gather_window<BS, SW, ES>(p, GlobalRows<BS>{p, 0}, lane, n_win, walk, off_lo, off_hi);

    auto issue = [&](int i, Vec16 *kk, Vec16 *vv) {
      const int64_t tile = window_tile_offset(off_lo, off_hi, i);
      const char *kb = p.k_pool + tile;
      const char *vb = p.v_pool + tile;
#pragma unroll
      for (int q4 = 0; q4 < NLD; ++q4) kk[q4] = load16(kb + lane_off[q4]);
#pragma unroll
      for (int q4 = 0; q4 < NLD; ++q4) vv[q4] = load16(vb + lane_off[q4]);
      // Keep the loads ahead of the arithmetic that follows in program order:
      // the scheduler would otherwise sink them below the current tile's work
      // and shorten the prefetch distance.
      __builtin_amdgcn_sched_barrier(0);
    };

    // Two register tiles in ping-pong.  The steady-state loop issues the next
    // tile's loads unconditionally, so the wait before a tile is consumed
    // covers that tile only and the prefetch stays in flight behind it,
    // across pair boundaries too.
    Vec16 ka[NLD], va[NLD], kb[NLD], vb[NLD];
    int i = 0;
    issue(0, ka, va);
    for (; i + 2 < n_win; i += 2) {
      issue(i + 1, kb, vb);
      consume(ka, va);
      issue(i + 2, ka, va);
      consume(kb, vb);
    }
    if (i + 2 == n_win) {
      issue(i + 1, kb, vb);
      consume(ka, va);
      consume(kb, vb);
    } else {
      consume(ka, va);
    }
  }
}

// Short contexts (up to 2 048 tokens at most, see decode_takes_pairs for the lines): with shares of a tile
// the split above turns them into partials that a second launch merges, 8 + 5 us of which the tiles themselves take
// two (4 sequences of up to 160 tokens, 12 heads of 64, fp32: 13.0 us, here 3.8).  Here a workgroup owns a whole pair:
// its eight waves take the pair's tiles in turn and merge through LDS (decode_pair.h); one launch, no workspace.  All types;
// the arithmetic is the vector-ALU kernel's (fp32 probabilities and sums).
// Bound by the chain of round trips: context length and table, tile, merge.
//
// APPEND: the step's append in the same launch (the layer call on 4 sequences of up to 192 tokens, 12 heads of 64,
// fp32: 11.6 -> 8.0 us).  Each workgroup stores the new rows of its pair and rotates its query rows.
struct PairAppend {
  const char *k_new, *v_new;
  const int64_t *slots;
  const int32_t *positions;  // rotary rows, or nullptr
  const float *cos_table, *sin_table;
  int64_t new_stride_bytes, num_slots, table_rows;
};

template <class E, int HD, int GT, bool APPEND>
struct PairRows {
  static constexpr bool kNew = APPEND, kLate = false;
  static constexpr int EPL = E::EPL, ES = sizeof(typename E::type);
  const DecodeKP &p;
  const PairAppend &n;
  const int seq, kvh, lane, col;
  // the step's new rows: lane j holds row j's slot, the wave this pair's own row (as it is stored)
  int64_t slot = -1;
  Vec16 own_k, own_v;
  __device__ __forceinline__ PairRows(const DecodeKP &p, const PairAppend &n, int seq, int kvh)
      : p(p), n(n), seq(seq), kvh(kvh), lane(threadIdx.x & (kWave - 1)), col(lane % (HD / EPL)) {}
  __device__ __forceinline__ int64_t table_row(int j) const {
    int64_t pos = n.positions[j];
    pos = pos < 0 ? 0 : pos;
    return (pos >= n.table_rows ? n.table_rows - 1 : pos) * (HD / 2) + col * (EPL / 2);
  }
  __device__ __forceinline__ int new_at() const { return (kvh * HD + col * EPL) * ES; }
  __device__ __forceinline__ Vec16 key(int j) const {
    const Vec16 k = load16(n.k_new + j * n.new_stride_bytes + new_at());
    if (n.positions == nullptr) return k;
    const int64_t at = table_row(j);
    return rotate_chunk<E>(k, n.cos_table + at, n.sin_table + at);
  }
  __device__ __forceinline__ Vec16 value(int j) const { return load16(n.v_new + j * n.new_stride_bytes + new_at()); }
  __device__ __forceinline__ bool sound() const { return true; }
  __device__ __forceinline__ void early() {
    if constexpr (APPEND) {
      if (lane < p.n_seqs) slot = n.slots[lane];
      if (slot >= n.num_slots) slot = -1;
      own_k = key(seq);
      own_v = value(seq);
    }
  }
  __device__ __forceinline__ void queries(Vec16 *qreg) const {
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      const int h = kvh * p.group + (g < p.group ? g : p.group - 1);
      qreg[g] = load16(p.q + (seq * p.q_stride_seq + (int64_t)h * HD + col * EPL) * ES);
      if constexpr (APPEND) {
        if (n.positions != nullptr) {
          const int64_t at = table_row(seq);
          qreg[g] = rotate_chunk<E>(qreg[g], n.cos_table + at, n.sin_table + at);
        }
      }
    }
  }
};

template <class E, int HD, int GT, bool APPEND>
__global__ __launch_bounds__(kPairWaves *kWave) void paged_decode_pair_kernel(const DecodeKP p, const PairAppend n) {
  using T = typename E::type;
  __shared__ PairShared<HD, GT> s;
  const int seq = blockIdx.y, kvh = blockIdx.x;
  PairRows<E, HD, GT, APPEND> rows(p, n, seq, kvh);
  const int tiles = walk_pair<E, HD, GT>(p, p.k_pool, p.v_pool, seq, kvh, threadIdx.x, s, rows);
  __syncthreads();
  T *orow = reinterpret_cast<T *>(p.out) + seq * p.out_stride_seq + (int64_t)kvh * p.group * HD;
  for (int o = threadIdx.x; o < p.group * HD; o += kPairWaves * kWave)
    orow[o] = E::narrow(tiles == 0 ? 0.f : pair_value(s, o / HD, o % HD));  // no visible token: zero rows
}

constexpr int kReduceThreads = 256;

// Where the split-K partials of one (sequence, pair) lie.  A pair's tiles in a
// row are a contiguous run of a phase's tile sequence, so the shares that
// touched it are first_tile / chunk .. last_tile / chunk and their partial ids
// follow.  With shared-prefix cohorts a sequence has two sources: its own row
// and its cohort's row of the shared phase, where it owns `group` of the matrix
// columns of one wave of each unit.
struct PartialList {
  int heads, head0;  // query heads of the pair
  int n_tiles;       // tiles behind the row (0: no visible token)
  int64_t n0, n_all;  // partials of source 0 (the cohort's row), of both
  int64_t base0, base1, stride0, stride1;  // slot of a source's first partial (column 0 of the pair), and between two
  // Slot of partial i, column g.
  __device__ __forceinline__ int64_t slot(int64_t i, int g) const {
    return g + (i < n0 ? base0 + i * stride0 : base1 + (i - n0) * stride1);
  }
};

__device__ __forceinline__ PartialList partial_list(const DecodeKP &p, int seq, int pair_in_seq) {
  PartialList r;
  const int COLS = p.gt;
  const int kvh = pair_in_seq / p.nsub;
  const bool cohorts = p.cohort_size > 1;
  int cohort = 0, col_sh = 0, wave_sh = 0;
  if (!cohorts) {
    const int sub = pair_in_seq - kvh * p.nsub;
    r.head0 = kvh * p.group + sub * COLS;
    r.heads = (p.group - sub * COLS < COLS) ? p.group - sub * COLS : COLS;
  } else {
    cohort = seq / p.cohort_size;
    const int u = seq - cohort * p.cohort_size;
    wave_sh = u / p.spw;                        // the wave of a unit that carries this member
    col_sh = (u - wave_sh * p.spw) * p.group;   // its first column there
    r.head0 = kvh * p.group;
    r.heads = p.group;
  }
  const int cum_own = p.cum_blocks[seq];
  const int nb_own = p.cum_blocks[seq + 1] - cum_own;
  const int cum_all = p.cum_blocks[p.n_seqs];
  int cum_sh = 0, nb_sh = 0, cum_sh_all = 0;
  if (cohorts) {
    cum_sh = p.cum_shared[cohort];
    nb_sh = p.cum_shared[cohort + 1] - cum_sh;
    cum_sh_all = p.cum_shared[p.n_cohorts];
  }
  r.n_tiles = nb_own + nb_sh;
  // source 0: the cohort's row of the shared phase, source 1: the sequence's
  // own row; an empty source has no partials.  Share w of a source left its
  // partial in slot (w + row and pair) of the own phase, resp. in the slots of
  // its unit's waves from shared_slot0 on.
  r.n0 = 0;
  r.base0 = r.stride0 = 0;
  if (nb_sh > 0) {
    const int64_t chunk = chunk_tiles(p, (int64_t)cum_sh_all * p.pairs_per_seq, phase_units(p, 1));
    const int64_t first = (int64_t)cum_sh * p.pairs_per_seq + (int64_t)pair_in_seq * nb_sh;
    const int64_t w_lo = first / chunk;
    r.n0 = (first + nb_sh - 1) / chunk - w_lo + 1;
    const int64_t unit_slot = w_lo + (int64_t)cohort * p.pairs_per_seq + pair_in_seq;
    r.base0 = (p.shared_slot0 + (unit_slot << p.unit_shift) + wave_sh) * COLS + col_sh;
    r.stride0 = (int64_t)COLS << p.unit_shift;
  }
  r.n_all = r.n0;
  r.base1 = 0;
  r.stride1 = COLS;
  if (nb_own > 0) {
    const int64_t chunk = chunk_tiles(p, (int64_t)cum_all * p.pairs_per_seq, phase_units(p, 0));
    const int64_t first = (int64_t)cum_own * p.pairs_per_seq + (int64_t)pair_in_seq * nb_own;
    const int64_t w_lo = first / chunk;
    r.n_all += (first + nb_own - 1) / chunk - w_lo + 1;
    r.base1 = (w_lo + (int64_t)seq * p.pairs_per_seq + pair_in_seq) * COLS;
  }
  return r;
}

// Four output dims of one head while partials are merged into them.
struct Merged {
  float m = kNegInf, l = 0.f;
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
  __device__ __forceinline__ void add(float pm, float pl, const float4 &pa) {
    if (pm == kNegInf) return;
    const float m_new = fmaxf(m, pm);
    const float keep = (m == kNegInf) ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
    const float wt = __builtin_amdgcn_exp2f(pm - m_new);
    l = __builtin_fmaf(pl, wt, l * keep);
    a.x = __builtin_fmaf(pa.x, wt, a.x * keep);
    a.y = __builtin_fmaf(pa.y, wt, a.y * keep);
    a.z = __builtin_fmaf(pa.z, wt, a.z * keep);
    a.w = __builtin_fmaf(pa.w, wt, a.w * keep);
    m = m_new;
  }
  // Partials first, first + step, ... of head column g, dims d .. d+3: fetched four at a time, all
  // loads of a batch independent and in flight together, whichever source they come from.
  template <int HD>
  __device__ __forceinline__ void add_all(const DecodeKP &p, const PartialList &pl, int64_t first, int64_t step, int g,
                                          int d) {
    constexpr int UB = 4;
    for (int64_t ib = first; ib < pl.n_all; ib += UB * step) {
      float2 ml[UB];
      float4 av[UB];
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        const int64_t i = ib + u * step < pl.n_all ? ib + u * step : pl.n_all - 1;
        const int64_t slot = pl.slot(i, g);
        ml[u] = *reinterpret_cast<const float2 *>(p.part_ml + slot * 2);
        av[u] = *reinterpret_cast<const float4 *>(p.part_acc + slot * HD + d);
      }
#pragma unroll
      for (int u = 0; u < UB; ++u)
        if (ib + u * step < pl.n_all) add(ml[u].x, ml[u].y, av[u]);
    }
  }
  template <class E>
  __device__ __forceinline__ void write(typename E::type *dst) const {
    const float inv = 1.f / l;
    dst[0] = E::narrow(a.x * inv);
    dst[1] = E::narrow(a.y * inv);
    dst[2] = E::narrow(a.z * inv);
    dst[3] = E::narrow(a.w * inv);
  }
};

// Combine the split-K partials of one pair (a KV head's query heads of one
// sequence).  grid = (pairs per sequence / pairs per workgroup, n_seqs).
// Traffic is (hd+2)*4 bytes per partial, three orders of magnitude below the
// K/V stream; what costs time here is the chain of dependent memory round
// trips, so the prefix sums are fetched together and every thread fetches up
// to four partials of its four output dims in one batch before it merges them
// (a typical pair has two to four partials: two round trips in all).
template <class E, int HD>
__global__ __launch_bounds__(kReduceThreads) void paged_decode_reduce_kernel(const DecodeKP p) {
  using T = typename E::type;
  constexpr int QPH = HD / 4;  // 4-dim groups per head row
  const int COLS = p.gt;
  // A pair keeps COLS * QPH threads busy; a workgroup takes as many pairs of
  // its sequence as fit (8 for MHA at hd 128), each on its own slice of threads.
  const int width = COLS * QPH < kReduceThreads ? COLS * QPH : kReduceThreads;
  const int per_wg = kReduceThreads / width;
  const int tid = threadIdx.x % width;
  const int pair_in_seq = blockIdx.x * per_wg + threadIdx.x / width;
  const int seq = blockIdx.y;
  if (pair_in_seq >= p.pairs_per_seq || threadIdx.x >= per_wg * width) return;
  const PartialList pl = partial_list(p, seq, pair_in_seq);
  T *orow = reinterpret_cast<T *>(p.out) + seq * p.out_stride_seq + (int64_t)pl.head0 * HD;
  if (pl.n_tiles == 0) {  // no visible token: zero rows
    for (int o = tid; o < pl.heads * HD; o += width) orow[o] = E::narrow(0.f);
    return;
  }
  // one wave covered all the sequence has for this pair and wrote the rows
  if (pl.n0 == 0 && pl.n_all == 1) return;
  for (int o = tid; o < pl.heads * QPH; o += width) {
    const int g = o / QPH;
    const int d = (o - g * QPH) * 4;
    Merged r;
    r.add_all<HD>(p, pl, 0, 1, g, d);
    r.write<E>(orow + g * HD + d);
  }
}

// The same for batches of few, long rows, whose pairs are cut over many waves
// (one sequence of 60 000 tokens: 112 partials per pair).  The kernel above
// walks them one batch of four after the other, a round trip each; here a
// workgroup belongs to ONE query head and its threads take the partials in
// slices (16 at head dim 128), which are merged through LDS at the end.
// grid = (hn, n_seqs).
//
// Measured, both launches of a call together, narrow / wide: 1 sequence of
// 60 001 tokens (32 / 8 heads, fp16, 112 partials per pair) 68.1 / 46.4 us, 1 of
// 4 096 (32 / 32 heads, 64 partials) 32.9 / 21.2 us, 4 of 8K-16K (32 / 8 heads,
// 28 partials) 47.0 / 41.8 us, 16 of 500-1 000 (16 partials) 23.3 / 21.3 us, 32 of
// 500-1 000 (8 partials, 1 024 workgroups) 29.5 / 31.4 us: hence the line at 12.
constexpr int kWideReduceThreads = 512;
constexpr int kWideReducePartials = 12;  // mean partials per pair from which this kernel is launched

template <class E, int HD>
__global__ __launch_bounds__(kWideReduceThreads) void paged_decode_wide_reduce_kernel(const DecodeKP p) {
  using T = typename E::type;
  constexpr int QPH = HD / 4;
  constexpr int SLICES = kWideReduceThreads / QPH;
  __shared__ __attribute__((aligned(16))) float s_acc[SLICES][HD];
  __shared__ float2 s_ml[SLICES];
  const int slice = threadIdx.x / QPH;
  const int d = (threadIdx.x - slice * QPH) * 4;
  const int seq = blockIdx.y;
  const int head = blockIdx.x;
  const int kvh = head / p.group;
  const int in_group = head - kvh * p.group;
  const int sub = p.cohort_size > 1 ? 0 : in_group / p.gt;
  const PartialList pl = partial_list(p, seq, kvh * p.nsub + sub);
  const int g = head - pl.head0;
  T *orow = reinterpret_cast<T *>(p.out) + seq * p.out_stride_seq + (int64_t)head * HD;
  if (pl.n_tiles == 0) {
    for (int o = threadIdx.x; o < HD; o += kWideReduceThreads) orow[o] = E::narrow(0.f);
    return;
  }
  if (pl.n0 == 0 && pl.n_all == 1) return;
  Merged r;
  r.add_all<HD>(p, pl, slice, SLICES, g, d);
  *reinterpret_cast<float4 *>(&s_acc[slice][d]) = r.a;
  if (d == 0) s_ml[slice] = make_float2(r.m, r.l);
  __syncthreads();
  if (slice != 0) return;
#pragma unroll
  for (int k = 1; k < SLICES; ++k)
    r.add(s_ml[k].x, s_ml[k].y, *reinterpret_cast<const float4 *>(&s_acc[k][d]));
  r.write<E>(orow + d);
}

// Waves of the main kernel that one GPU holds at once, per kernel variant.
template <class E, int HD, int GT, int BS, int NW>
int resident_workgroups() {
  static const int per_cu = [] {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, paged_decode_kernel<E, HD, GT, BS, NW>,
                                                     NW * kWave, 0) != hipSuccess || n < 1)
      n = 1;
    return n;
  }();
  return per_cu * device_cu_count();
}

template <class E, int HD>
int launch_reduce(const DecodeKP &kp, hipStream_t stream) {
  // Partials of a pair, when the rows are equally long: its share of the waves, one tile each at least.
  const int64_t shares = kp.n_waves / ((int64_t)kp.n_seqs * kp.pairs_per_seq);
  if ((shares < kp.max_ctx / 16 ? shares : kp.max_ctx / 16) >= kWideReducePartials) {
    hipLaunchKernelGGL((paged_decode_wide_reduce_kernel<E, HD>), dim3(kp.hn, kp.n_seqs), dim3(kWideReduceThreads), 0,
                       stream, kp);
    return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
  }
  const int width = kp.gt * (HD / 4) < kReduceThreads ? kp.gt * (HD / 4) : kReduceThreads;
  const int per_wg = kReduceThreads / width;  // pairs per workgroup, as the kernel derives it
  hipLaunchKernelGGL((paged_decode_reduce_kernel<E, HD>), dim3((kp.pairs_per_seq + per_wg - 1) / per_wg, kp.n_seqs),
                     dim3(kReduceThreads), 0, stream, kp);
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

// fp32 pools: the vector-ALU main kernel, one instantiation per group size.
template <class E, int HD, int GT>
void launch_valu_main(DecodeKP &kp, hipStream_t stream) {
  constexpr int BS = 16;
  constexpr int NW = kDecodeWavesPerWorkgroup;
  int wgs = resident_workgroups<E, HD, GT, BS, NW>();
  if (wgs * NW > kp.max_waves) wgs = kp.max_waves / NW;
  kp.n_waves = wgs * NW;
  hipLaunchKernelGGL((paged_decode_kernel<E, HD, GT, BS, NW>), dim3(wgs), dim3(NW * kWave), 0, stream, kp);
}

// Tiles in turn of the pair kernel's waves on the longest row.
int64_t pair_rounds(const DecodeKP &kp) { return ((int64_t)kp.max_ctx + 16 * kPairWaves - 1) / (16 * kPairWaves); }

// Whether a call is the pair kernel's.  us of the split (main kernel and reduce) / of the pair kernel, contexts up to
// 48, 160, 300, 600, 1 200 tokens:
//   fp32, 12 / 12 heads of 64, 4 sequences     9.8 / 3.1   13.0 / 3.8   15.6 / 4.3   19.3 / 5.5   27.9 / 8.1
//   fp32, 32 / 32 of 128, 4                   11.6 / 3.7   14.1 / 5.0   18.9 / 7.7   26.8 / 13.8  35.6 / 22.4
//   bf16, 32 / 32 of 128, 4                   11.0 / 3.6   13.0 / 4.5   14.8 / 5.1   20.2 / 8.0   24.6 / 13.9
//   bf16, 16 / 16 of 64, 40                   14.4 / 4.7   18.3 / 5.6   22.3 / 9.4
//   bf16, 32 / 8 of 128, 4                    10.2 / 6.4   13.0 / 8.4   15.2 / 10.1  19.7 / 14.3  18.2 / 21.3
//   bf16, 32 / 8 of 128, 40                   12.2 / 11.8  16.0 / 15.2  19.9 / 20.9
//   bf16, 28 / 4 of 128, 4                    10.1 / 10.4  13.2 / 14.1  15.2 / 17.1
// Larger batches, contexts of 20-64, 20-200, 17-512, 50-1 000 and 30-2 000 tokens, split / this kernel:
//   bf16, 16 / 16 of 64, 64      19.7 / 7.4   22.1 / 10.1  30.7 / 19.3   42.0 / 31.6    67.8 / 58.1
//   bf16, 16 / 16 of 64, 233     23.9 / 19.4  39.9 / 28.4  67.6 / 51.6   111.5 / 95.2   200.0 / 180.6
//   bf16, 32 / 32 of 128, 64     20.6 / 18.7  34.1 / 29.0  64.0 / 56.6   110.8 / 105.2  211.6 / 197.8
//   bf16, 32 / 32 of 128, 233    49.0 / 54.7  98.9 / 88.0  201.1 / 181.9 363.7 / 349.5  678.9 / 669.3
//   fp32, 32 / 32 of 128, 64     31.2 / 33.5  56.8 / 55.9  112.9 / 102.9 201.7 / 193.1  393.7 / 379.8
//   fp32, 32 / 32 of 128, 233    83.3 / 109   179 / 182    380 / 350     708 / 681
//   bf16, 8 / 4 of 64, 233       20.0 / 11.4  22.6 / 13.6  30.2 / 20.0   41.3 / 32.5    56.5 / 56.6
//   bf16, 16 / 8 of 128, 4       13.3 / 6.5   14.7 / 7.6   16.1 / 9.3    17.1 / 13.4    16.4 / 20.3
//   bf16, 16 / 8 of 128, 256     21.3 / 22.9  35.7 / 33.7  68.0 / 58.9   114.3 / 106.8  204.7 / 199.2
//   bf16, 16 / 4 of 64, 4        12.0 / 8.1   13.7 / 9.9   14.6 / 11.6   19.6 / 15.2    16.3 / 22.4
//   bf16, 16 / 4 of 64, 256      20.7 / 18.8  23.3 / 22.8  32.2 / 30.3   44.1 / 42.2    64.5 / 66.8
// and batches with one long row among rows of 20 tokens, which the split balances and a workgroup walks alone (1 000, 2 000):
//   bf16, 16 / 16 of 64, 4 and 233       20.6 / 7.4, 21.0 / 10.4 and 26.7 / 18.0, 27.7 / 20.7
//   bf16, 32 / 32 of 128, 4 and 64       16.9 / 10.9, 18.8 / 16.0 and 24.9 / 19.3, 29.3 / 30.4
//   fp32, 32 / 32 of 128, 4              20.1 / 15.8, 25.2 / 42.3
// So the rows a workgroup walks are limited by their bytes (a round is 128 tokens), and the pairs by theirs: tens of
// thousands of short rows start more workgroups than the split does.  Grouped heads cost this kernel vector work for
// each head, hence lower limits, and none from five heads on.
bool decode_takes_pairs(const DecodeKP &kp, int hd, int row_bytes) {
  if (kp.cohort_size != 1 || kp.key_mask != nullptr || kp.min_chunk > 1 || kp.max_ctx <= 0 || kp.group > 4) return false;
  const int64_t rounds = pair_rounds(kp);
  const int64_t pairs = (int64_t)kp.n_seqs * kp.pairs_per_seq;
  if (rounds > 16 || kp.n_seqs > 65535) return false;
  if (kp.group == 1) return rounds * row_bytes <= 4096 && pairs * row_bytes < (rounds == 1 ? 1 << 20 : 2 << 20);
  if (kp.group == 2) return rounds * row_bytes <= 2048 && pairs * row_bytes < 1 << 19;
  if (hd <= 64) return rounds <= 8 && pairs <= 2 * device_cu_count();
  return rounds <= 2 && pairs <= device_cu_count();
}

// Whether the append rides on the pair kernel's launch.  It saves a launch of about a microsecond and costs each workgroup
// the comparison of its tiles with all new slots: worth it while a CU has one workgroup, not with two.  us of one launch / of
// two (append, attention), by pairs (KV heads times sequences), contexts up to 250, 500, 1 000 and 2 000 tokens:
//   fp32, 12 / 12 heads of 64             48    5.0 / 6.2    6.0 / 7.2    8.1 / 9.0    15.0 / 16.0
//                                        192    5.3 / 6.3    7.7 / 8.5   13.9 / 14.6   22.3 / 23.2
//                                        384   10.7 / 9.5   16.5 / 16.3  26.2 / 25.9   52.4 / 51.2
//   bf16, 16 / 16 of 64, rotary           64    5.5 / 6.4    6.3 / 7.1    7.8 / 8.5    10.8 / 10.9
//                                        256    6.1 / 6.5    6.6 / 7.3   13.0 / 12.8   18.6 / 18.5
//                                        512    8.8 / 7.7   15.5 / 13.8  21.7 / 20.6   34.7 / 33.5
//   bf16, 8 / 8 of 128, rotary            32    6.3 / 7.1    7.6 / 8.2   10.2 / 10.2   15.1 / 14.1
//                                        256    7.0 / 7.4   13.2 / 13.3  19.7 / 20.0   32.4 / 32.4
//                                        512   14.5 / 13.2  21.2 / 19.5  33.9 / 31.5   79.0 / 69.5
// Grouped heads rotate a query row for each of them, in every wave: fewer pairs, fewer rounds.
//   bf16, 8 / 4 of 64, rotary             16    7.1 / 7.7    8.3 / 8.9   10.6 / 10.7   15.2 / 14.6
//                                        128    7.5 / 7.9    8.7 / 9.0   11.8 / 11.0   18.1 / 16.6
//                                        256    8.0 / 8.1    9.8 / 9.6   15.6 / 14.9   22.0 / 21.5
//   bf16, 16 / 8 of 128, rotary           32    7.8 / 8.6    9.7 / 10.3  13.6 / 13.8
//                                        128    8.1 / 8.6   10.0 / 10.4  16.6 / 15.8
//                                        512   20.5 / 15.0  26.8 / 21.5  38.8 / 34.2
//   fp16, 8 / 2 of 64, rotary              8   10.3 / 10.5  12.2 / 12.2  16.1 / 15.9
//                                         64   10.5 / 10.6  12.4 / 12.4  16.3 / 16.0
//   bf16, 16 / 4 of 64, rotary           256   11.6 / 11.2  14.0 / 13.2  21.8 / 19.1
bool append_joins_pairs(const DecodeKP &kp, int hd) {
  const int64_t rounds = pair_rounds(kp), pairs = (int64_t)kp.n_seqs * kp.pairs_per_seq, cus = device_cu_count();
  if (kp.n_seqs > kPairAppendRows || pairs > cus) return false;
  if (kp.group == 1) return rounds * hd <= 1024;
  if (kp.group == 2) return rounds <= 8 && pairs * rounds <= 2 * cus;
  return rounds <= 4 && pairs * rounds <= cus && 2 * pairs <= cus;
}

template <class E, int HD, bool APPEND>
int launch_pairs(const DecodeKP &kp, const PairAppend &rows, hipStream_t stream) {
  const dim3 grid(kp.pairs_per_seq, kp.n_seqs), block(kPairWaves * kWave);
  if (kp.group == 1)
    hipLaunchKernelGGL((paged_decode_pair_kernel<E, HD, 1, APPEND>), grid, block, 0, stream, kp, rows);
  else if (kp.group == 2)
    hipLaunchKernelGGL((paged_decode_pair_kernel<E, HD, 2, APPEND>), grid, block, 0, stream, kp, rows);
  else
    hipLaunchKernelGGL((paged_decode_pair_kernel<E, HD, 4, APPEND>), grid, block, 0, stream, kp, rows);
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

template <class E, int HD>
int launch_group(DecodeKP &kp, int dtype, const AppendRows *rows, hipStream_t stream) {
  const bool pairs = decode_takes_pairs(kp, HD, HD * (int)sizeof(typename E::type));
  if (rows != nullptr) {  // with the append: only in one launch
    if (!pairs || !append_joins_pairs(kp, HD) || kp.num_blocks * kp.tiles_per_block >= (int64_t)1 << 31)
      return IC_ERR_UNSUPPORTED;
    PairAppend n;
    n.k_new = (const char *)rows->k_new, n.v_new = (const char *)rows->v_new;
    n.slots = rows->slots, n.positions = rows->cos_table != nullptr ? rows->positions : nullptr;
    n.cos_table = rows->cos_table, n.sin_table = rows->sin_table;
    n.new_stride_bytes = rows->new_stride_token * (int64_t)sizeof(typename E::type);
    n.num_slots = kp.num_blocks * kp.tiles_per_block * 16;
    n.table_rows = rows->table_rows;
    return launch_pairs<E, HD, true>(kp, n, stream);
  }
  if (pairs) return launch_pairs<E, HD, false>(kp, PairAppend{}, stream);
  if constexpr (sizeof(typename E::type) == 2) {
    // 16-bit element types: the matrix-core kernel, whatever the group size.
    if (!launch_decode_mfma_main(kp, dtype, HD, stream)) return IC_ERR_UNSUPPORTED;
  } else {
    if (kp.cohort_size != 1) return IC_ERR_UNSUPPORTED;
    switch (kp.gt) {
      case 1: launch_valu_main<E, HD, 1>(kp, stream); break;
      case 2: launch_valu_main<E, HD, 2>(kp, stream); break;
      case 3: launch_valu_main<E, HD, 3>(kp, stream); break;
      case 4: launch_valu_main<E, HD, 4>(kp, stream); break;
      case 5: launch_valu_main<E, HD, 5>(kp, stream); break;
      case 6: launch_valu_main<E, HD, 6>(kp, stream); break;
      case 7: launch_valu_main<E, HD, 7>(kp, stream); break;
      default: launch_valu_main<E, HD, 8>(kp, stream); break;
    }
  }
  return launch_reduce<E, HD>(kp, stream);
}

template <class E>
int launch_hd(DecodeKP &kp, int hd, int dtype, const AppendRows *rows, hipStream_t stream) {
  switch (hd) {
    case 32: return launch_group<E, 32>(kp, dtype, rows, stream);
    case 64: return launch_group<E, 64>(kp, dtype, rows, stream);
    case 128: return launch_group<E, 128>(kp, dtype, rows, stream);
    default: return IC_ERR_UNSUPPORTED;
  }
}

}  // namespace

int launch_paged_decode(const DecodeArgs &a, hipStream_t stream) {
  // The kernel loads whole 16-token tiles, so a pool block must hold a whole
  // number of them (a tile never straddles the end of a block).
  if (a.pool.block_size % 16 != 0) return IC_ERR_UNSUPPORTED;
  DecodeKP kp;
  kp.q = (const char *)a.q;
  kp.k_pool = (const char *)a.k_pool;
  kp.v_pool = (const char *)a.v_pool;
  kp.block_tables = a.block_tables;
  kp.context_lens = a.context_lens;
  kp.out = (char *)a.out;
  kp.cum_blocks = a.cum_blocks;
  kp.part_ml = a.part_ml;
  kp.part_acc = a.part_acc;
  kp.q_stride_seq = a.q_stride_seq;
  kp.out_stride_seq = a.out_stride_seq;
  kp.stride_block = a.pool.stride_block;
  kp.stride_head = a.pool.stride_head;
  kp.stride_token = a.pool.stride_token;
  kp.bt_stride = a.block_table_stride;
  kp.num_blocks = a.pool.num_blocks;
  kp.n_seqs = a.n_seqs;
  kp.hn = a.hn;
  kp.group = a.hn / a.gn;
  const DecodeLayout lay = decode_layout(a.n_seqs, a.hn, a.gn, a.cohort_size);
  if (!lay.ok) return IC_ERR_UNSUPPORTED;
  kp.nsub = lay.nsub;
  kp.gt = lay.cols;
  kp.pairs_per_seq = a.gn * lay.nsub;
  kp.cohort_size = a.cohort_size > 1 ? a.cohort_size : 1;
  kp.cohort_shared = a.cohort_size > 1 ? a.cohort_shared_blocks : nullptr;
  kp.n_cohorts = lay.n_cohorts;
  kp.spw = lay.spw;
  kp.unit_shift = lay.unit_shift;
  kp.cum_shared = a.cum_blocks + a.n_seqs + 1;
  kp.shared_slot0 = a.shared_slot0;
  kp.max_ctx = a.max_context_len;
  kp.n_waves = 0;
  kp.max_waves = a.max_waves > 0 && a.max_waves < kMaxDecodeWaves ? a.max_waves : kMaxDecodeWaves;
  kp.min_chunk = (a.min_chunk_tokens + 15) / 16;
  kp.tiles_per_block = a.pool.block_size / 16;
  kp.scale_log2e = a.scale * 1.4426950408889634f;
  kp.key_mask = a.key_mask;
  kp.key_mask_stride_seq = a.key_mask_stride_seq;
  kp.key_mask_stride_head = a.key_mask_stride_head;
  if (a.key_mask != nullptr && a.dtype != IC_DTYPE_F32) return IC_ERR_UNSUPPORTED;
  switch (a.dtype) {
    case IC_DTYPE_BF16: return launch_hd<Bf16>(kp, a.hd, a.dtype, a.rows, stream);
    case IC_DTYPE_F16: return launch_hd<F16>(kp, a.hd, a.dtype, a.rows, stream);
    case IC_DTYPE_F32: return launch_hd<F32>(kp, a.hd, a.dtype, a.rows, stream);
    default: return IC_ERR_UNSUPPORTED;
  }
}

}  // namespace ic
