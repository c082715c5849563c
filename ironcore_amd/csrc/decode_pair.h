// The walk of one workgroup over one (sequence, KV head) pair of a decode step, for short contexts: eight waves take the
// pair's 16-token tiles in turn (a wave's table entries come in one load, one per lane: at most 64 tiles), keep a running
// softmax each and merge through LDS.  Vector arithmetic, fp32 probabilities and sums, all types.  Used by
// paged_decode_pair_kernel (paged_decode.hip) and by the attention tasks of step_stack_kernel (step_stack.hip).
//
// With new rows (Rows::kNew) the step's append is part of the walk: the workgroup stores its pair's new rows.  A new row
// may be visible to any sequence (rows of one sequence at several positions, shared blocks), and another workgroup may
// store it sooner or later than it is read here, so what a tile holds in a slot of this step is always taken from the new
// rows: lane j has row j's slot (64 rows at most), and a tile compares its id with all of them at once.
#pragma once

#include "decode_common.h"

namespace ic {
namespace decode {

constexpr int kPairWaves = 8;
constexpr int kPairAppendRows = kWave;

template <int HD, int GT>
struct PairShared {
  __attribute__((aligned(16))) float acc[kPairWaves][GT][HD];
  float m[kPairWaves][GT], l[kPairWaves][GT];
};

// Leaves the waves' sums in `s` and returns the number of tiles; the caller's barrier comes next.  `rows` hands over the query rows and, with kNew, the
// step's new rows: the slots, a lane a row, the pair's own row as it is stored (if it is sound()), any other row by key(j) and
// value(j), all in the lane's chunk.  kLate: the queries (and the own row) are asked for once the first two tiles are on their way.
template <class E, int HD, int GT, class Rows>
__device__ __forceinline__ int walk_pair(const DecodeKP &p, const char *k_pool, const char *v_pool, int seq, int kvh,
                                         int thread, PairShared<HD, GT> &s, Rows &rows) {
  constexpr int EPL = E::EPL;
  constexpr int ES = sizeof(typename E::type);
  constexpr int LPR = HD / EPL;     // lanes sharing one token row
  constexpr int RPL = kWave / LPR;  // token rows per load instruction
  constexpr int BS = 16;
  constexpr int NLD = BS / RPL;     // load instructions per tile
  const int lane = thread & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(thread / kWave);
  const int col = lane % LPR;
  const int rowg = lane / LPR;

  int ctx = p.context_lens[seq];
  ctx = ctx < p.max_ctx ? ctx : p.max_ctx;
  ctx = ctx < 0 ? 0 : ctx;
  const int tiles = (ctx + BS - 1) / BS;
  const int mine = __builtin_amdgcn_readfirstlane(tiles > wave ? (tiles - wave + kPairWaves - 1) / kPairWaves : 0);
  rows.early();
  // lane r: byte offset of this wave's tile of round r, and the tile's number in the pool (lanes past the last round: the last
  // one's).  Nothing here depends on the lane's number but its operands: behind a branch of some lanes the compiler has put
  // registers into scratch before it switched the other lanes on again, and a wave without tiles then lost its lanes' numbers.
  int64_t tile_off = 0;
  int tile_id = -1;
  if (mine > 0) {
    const int tile = wave + (lane < mine ? lane : mine - 1) * kPairWaves;
    const int blk = tile / p.tiles_per_block;
    int64_t phys = p.block_tables[seq * p.bt_stride + blk];
    // A corrupt table entry must not become an out-of-pool address.
    phys = phys < 0 ? 0 : phys;
    phys = phys >= p.num_blocks ? p.num_blocks - 1 : phys;
    tile_off = (phys * p.stride_block + kvh * p.stride_head +
                (int64_t)(tile - blk * p.tiles_per_block) * BS * p.stride_token) * ES;
    if constexpr (Rows::kNew) tile_id = (int)(phys * p.tiles_per_block) + tile - blk * p.tiles_per_block;
  }
  Vec16 qreg[GT];
  if constexpr (!Rows::kLate) rows.queries(qreg);
  uint32_t lane_off[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) lane_off[i] = (uint32_t)(((i * RPL + rowg) * p.stride_token + col * EPL) * ES);

  float m[GT], l[GT], acc[GT][EPL];
#pragma unroll
  for (int g = 0; g < GT; ++g) {
    m[g] = kNegInf;
    l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[g][e] = 0.f;
  }
  auto issue = [&](int r, Vec16 *kk, Vec16 *vv) __attribute__((always_inline)) {
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)tile_off, r);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)((uint64_t)tile_off >> 32), r);
    const int64_t at = (int64_t)(((uint64_t)hi << 32) | lo);
#pragma unroll
    for (int i = 0; i < NLD; ++i) kk[i] = load16(k_pool + at + lane_off[i]);
#pragma unroll
    for (int i = 0; i < NLD; ++i) vv[i] = load16(v_pool + at + lane_off[i]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto consume = [&](int r, Vec16 *kk, Vec16 *vv) __attribute__((always_inline)) {
    if constexpr (Rows::kNew) {
      const int id = __builtin_amdgcn_readlane(tile_id, r);
      const int64_t slot = rows.slot;
      uint64_t found = __ballot(slot >= 0 && (int)(slot / BS) == id);
      for (; found != 0; found &= found - 1) {
        const int j = __builtin_ctzll(found);
        const int token = __builtin_amdgcn_readlane((int)(slot % BS), j);
        Vec16 k = rows.own_k, v = rows.own_v;
        if (j != seq) k = rows.key(j), v = rows.value(j);
#pragma unroll
        for (int i = 0; i < NLD; ++i)
          if (token == i * RPL + rowg) kk[i] = k, vv[i] = v;
      }
    }
    float sc[GT][NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i)
#pragma unroll
      for (int g = 0; g < GT; ++g) sc[g][i] = group_sum<LPR>(E::dot(kk[i], qreg[g], 0.f)) * p.scale_log2e;
    const int tok0 = (wave + r * kPairWaves) * BS;
    if (tok0 + BS > ctx) {  // the sequence's last tile may be partly filled
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        if (tok0 + i * RPL + rowg >= ctx) {
#pragma unroll
          for (int g = 0; g < GT; ++g) sc[g][i] = kNegInf;
          vv[i] = Vec16{{0u, 0u, 0u, 0u}};
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
      for (int i = 0; i < NLD; ++i) mx = fmaxf(mx, sc[g][i]);
      const float ms = (mx == kNegInf) ? 0.f : mx;
      const float alpha = __builtin_amdgcn_exp2f(m[g] - ms);
      float pr[NLD];
      float ps = 0.f;
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        pr[i] = __builtin_amdgcn_exp2f(sc[g][i] - ms);
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
  };
  Vec16 ka[NLD], va[NLD], kb[NLD], vb[NLD];
  if (mine > 0) issue(0, ka, va);
  if constexpr (Rows::kLate) {
    if (mine > 0) issue(mine > 1 ? 1 : 0, kb, vb);
    rows.queries(qreg);
  }
  if constexpr (Rows::kNew) {
    // the last wave has the fewest tiles; K from its first row of lanes, V from the second
    const int64_t to = ((int64_t)__builtin_amdgcn_readlane((uint32_t)((uint64_t)rows.slot >> 32), seq) << 32) |
                       (uint32_t)__builtin_amdgcn_readlane((uint32_t)rows.slot, seq);
    if (wave == kPairWaves - 1 && to >= 0 && rows.sound() && rowg < 2) {
      const int64_t blk = (uint64_t)to / (uint32_t)(p.tiles_per_block * BS);
      const int64_t at = blk * p.stride_block + kvh * p.stride_head + (to - blk * p.tiles_per_block * BS) * p.stride_token;
      Vec16 own;  // (word by word: a choice between two members would put `rows` into scratch)
#pragma unroll
      for (int i = 0; i < 4; ++i) own.w[i] = rowg == 0 ? (uint32_t)rows.own_k.w[i] : (uint32_t)rows.own_v.w[i];
      store16(const_cast<char *>(rowg == 0 ? k_pool : v_pool) + (at + col * EPL) * ES, own);
    }
  }
  for (int r = 0; r < mine; r += 2) {
    if (!Rows::kLate || r > 0) issue(r + 1 < mine ? r + 1 : r, kb, vb);
    consume(r, ka, va);
    if (r + 1 >= mine) break;
    issue(r + 2 < mine ? r + 2 : r + 1, ka, va);
    consume(r + 1, kb, vb);
  }

  // ---- merge: the row groups of a wave by exchange, the waves through LDS ----------------------
#pragma unroll
  for (int g = 0; g < GT; ++g) {
    float mx = m[g];
#pragma unroll
    for (int off = LPR; off < kWave; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
    const float w = (m[g] == kNegInf) ? 0.f : __builtin_amdgcn_exp2f(m[g] - mx);
    float ls = l[g] * w;
#pragma unroll
    for (int off = LPR; off < kWave; off <<= 1) ls += __shfl_xor(ls, off, kWave);
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      float a = acc[g][e] * w;
#pragma unroll
      for (int off = LPR; off < kWave; off <<= 1) a += __shfl_xor(a, off, kWave);
      if (rowg == 0) s.acc[wave][g][col * EPL + e] = a;
    }
    if (lane == 0) {
      s.m[wave][g] = mx;
      s.l[wave][g] = ls;
    }
  }
  return tiles;
}

// Output element d of query head g, once the waves' sums are there (of a pair that has tiles).
template <int HD, int GT>
__device__ __forceinline__ float pair_value(const PairShared<HD, GT> &s, int g, int d) {
  float mx = kNegInf;
#pragma unroll
  for (int v = 0; v < kPairWaves; ++v) mx = fmaxf(mx, s.m[v][g]);
  float sum = 0.f, a = 0.f;
#pragma unroll
  for (int v = 0; v < kPairWaves; ++v) {
    const float w = s.m[v][g] == kNegInf ? 0.f : __builtin_amdgcn_exp2f(s.m[v][g] - mx);
    sum = __builtin_fmaf(s.l[v][g], w, sum);
    a = __builtin_fmaf(s.acc[v][g][d], w, a);
  }
  return a / sum;
}

}  // namespace decode
}  // namespace ic
