// Chunked prefill for 16-bit pools, the kernel for short work: chunks of a few
// rows to a few hundred, and batches too small to fill the GPU with the
// 256-row workgroups of paged_prefill.hip.
//
// Same contract and the same arithmetic per tile (K/V tiles of 64 tokens
// straight into swizzled LDS, S^T = K Q^T and O^T += V^T P^T on
// v_mfma_f32_32x32x16, lazy reference maximum).  What differs is the shape:
//
//  * A workgroup is 4 waves, each owning a WAVE BLOCK of 32 query rows of one
//    head.  The blocks of a KV head's G query heads are numbered through
//    (ceil(C / 32) per head), and a workgroup takes four neighbouring ones, so
//    short chunks of several heads share a workgroup and its K/V tiles: 13 rows
//    x 7 heads are two workgroups, not seven with 5 % of their rows in use.
//    Blocks are numbered row block by row block, the heads of a row block side by
//    side: the waves of a workgroup reach about equally far (a packed mask's
//    lists belong to a head's rows: there, and with DIRECT, head by head).
//  * Chunks of unequal length that fill the chip more than once: workgroups are numbered over all
//    sequences, the longest sweep first (by_sweep below), KV heads round the XCDs.
//  * Every wave stages a 16-row group of K AND of V of each tile, into two
//    buffers (a third gained nothing); one barrier per tile.  64 KiB of LDS at head dim 128, 32 KiB at 64:
//    two, resp. four, workgroups share a CU, and what the two-sided schedule of
//    the long kernel arranges inside a workgroup (matrix work beside vector
//    work, loads behind both) comes here from neighbours that are at other
//    points of their sweeps, start and end included, which is most of a short
//    sweep's life.
//  * Grids that leave one workgroup to a CU run it with two groups of four waves
//    (TG = 2) on the same query rows, which take the tiles in turn and merge
//    their sums through LDS at the end: half the tiles one after the other.
//
//  * PACKED: a general mask as mask_pack.hip leaves it.  The sweep visits the tiles
//    of the query tile's list; a wave skips the ones its 32 rows do not see and
//    applies the words (fetched with the tile, 256 bytes per wave) only where they
//    are mixed.  2 x 1 024 tokens in packed documents, 16 heads of 64: 149 us with
//    the byte mask of the long kernel (32 byte loads per lane and tile, every tile
//    walked), 11.9 us here, launch to launch.
//
//  * In full grids, and with rotary from a few rows on, query rows and outputs move as whole rows of a head and change places in LDS: as
//    the MFMA lays them out a load touched 32 cache lines for 1 KiB, rotary tables likewise (query rows ready after 3.8
//    instead of 5.3 us of a workgroup's 17; 80 sequences of 129 tokens, 12 heads of 64: 20.8 -> 18.8 us).  The others
//    (DIRECT, prefill_rows_direct) load and store them as they are needed.
//
// Bound by the latency of a tile (load, two products and a softmax in one wave's
// instruction stream, about 1 us at head dim 128) at the sizes it is for; 80
// sequences of 129 tokens, 12 heads of 64, without a cache: 24.1 -> 19.8 us; 9
// prompts of 3-701 tokens, 28 / 4 heads of 128: 32.0 -> 24.3 us; 67 of 18 tokens,
// 32 / 8 heads of 128: 41.1 -> 12.5 us (the long kernel -> this one).
#include "prefill_common.h"
#include "../../include/ironcore_paged.h"

namespace ic {
namespace prefill {

namespace {

constexpr int kShortWaves = 4;  // wave blocks per workgroup
constexpr int kBN = 64;         // tokens per K/V tile

constexpr int kShortBuffers = 2;  // LDS buffers per pool and tile group

// Chunks of unequal length, at most one sequence per lane: workgroup `index` of a KV head, numbered over the sequences by
// the tiles it has to walk, most first.  Workgroup w of a sequence walks more tiles than its workgroup w - 1, so the number
// that walk more than t tiles is a formula, and a binary search over t finds the index's t, then its sequence.
// False: past the last one.  v0: its first wave block.
//
// 9 prompts of 3-701 tokens, 28 / 4 heads of 128, rotary: numbered sequence by sequence (units of a KV head on an
// XCD) the XCDs had 82 to 102 workgroups, and the longest of a middle sequence began when half the launch was over
// (the layer call 51.7 -> 49.2 us; with whole rows of queries and outputs, below, 40.4).
__device__ __forceinline__ bool pick_by_sweep(const PrefillKP &p, int index, int &seq, int &q_lo, int &L, int &C, int &v0) {
  const int n_seqs = p.n_units / p.gn, ln = threadIdx.x & (kWave - 1), group = p.group;
  const bool in = ln < n_seqs;
  const int lo = in ? chunk_begin(p, ln) : 0, chunk = in ? chunk_end(p, ln) - lo : 0;
  int len = in ? p.context_lens[ln] : 0;
  len = len < 0 ? 0 : len;
  const int rows = p.causal && chunk > len ? len : chunk;
  const int blocks = rows > 0 ? (rows + 31) >> 5 : 0;
  const int wgs = (blocks * group + kShortWaves - 1) / kShortWaves;
  const int prefix = len - rows;
  // workgroups of this lane's sequence that walk more than t tiles (t == 0: all of them)
  auto longer = [&](int t) {
    if (t == 0) return wgs;
    const int keys = t * kBN;
    if (keys >= len) return 0;
    if (!p.causal) return wgs;
    const int block = keys > prefix ? (keys - prefix) >> 5 : 0;  // the first that sees past `keys`
    const int first = (block * group) / kShortWaves;             // the workgroup that holds it (and rows of no later block)
    return wgs > first ? wgs - first : 0;
  };
  // (counts are exact in fp32; up to 16 sequences stay inside a row of lanes, whose exchanges are vector instructions)
  auto total = [&](int t) {
    const float n = (float)longer(t);
    return __builtin_amdgcn_readfirstlane((int)(n_seqs <= 16 ? group_sum<16>(n) : group_sum<kWave>(n)));
  };
  if (index >= total(0)) return false;
  int above = 1;  // total(t) > index >= total(above)
  while (total(above) > index) above *= 2;
  int t = above >> 1;
  while (above - t > 1) {
    const int mid = (t + above) >> 1;
    if (total(mid) > index)
      t = mid;
    else
      above = mid;
  }
  const int beyond = longer(t + 1), here = longer(t) - beyond;
  int rest = index - total(t + 1);
  seq = 0;
  for (int j = 0; j < n_seqs; ++j) {
    const int n = __builtin_amdgcn_readlane(here, j);
    if (rest < n) {
      seq = j;
      break;
    }
    rest -= n;
  }
  q_lo = __builtin_amdgcn_readlane(lo, seq);
  L = __builtin_amdgcn_readlane(len, seq);
  C = __builtin_amdgcn_readlane(chunk, seq);
  v0 = (__builtin_amdgcn_readlane(wgs - beyond, seq) - 1 - rest) * kShortWaves;
  return true;
}

// DIRECT: query rows and outputs move as the MFMA lays them out, and the row blocks of a head side by side (see
// prefill_rows_direct).
template <class M, int HD, bool SINGLE, int TG, bool PACKED, bool DIRECT>
__global__ __launch_bounds__(TG *kShortWaves *kWave) __attribute__((amdgpu_waves_per_eu(HD == 128 ? 2 : 4)))
void paged_prefill_short_kernel(const PrefillKP p) {
  constexpr int KS = HD / 16;      // k-steps of the QK contraction
  constexpr int OB = HD / 32;      // 32-wide blocks of the output head dim
  constexpr int TB = kBN / 32;     // 32-token blocks per tile
  constexpr int CPR = HD / 8;      // 16-byte chunks per token row
  constexpr int WR = kWave / CPR;  // token rows one load instruction of a wave covers
  constexpr int NST = 16 / WR;     // loads per lane, pool and staged tile
  constexpr int ROWB = HD * 2;

  constexpr int NB = kShortBuffers;
  constexpr int TILEB = kBN * ROWB;  // bytes of a tile in one pool

  // [tile group][pool][buffer][tile]; after the sweep the second group hands its sums over in it
  constexpr int kMergeBytes = TG > 1 ? kShortWaves * (OB * 16 + 2) * kWave * 4 : 0;
  constexpr int kTileBytes = TG * 2 * NB * TILEB;
  __shared__ __attribute__((aligned(1024))) char s_tiles[kTileBytes > kMergeBytes ? kTileBytes : kMergeBytes];
  __shared__ uint64_t s_words[PACKED ? TG * kShortWaves * NB * 32 : 1];  // packed mask: a wave's words of its tiles

  // XCD-aware placement as in the long kernel: the workgroups of one (sequence, KV head) unit get ids
  // that differ by a multiple of 8.
  int seq, q_lo, L, C, kvh, v0 = 0, slice = 0, r = 0;
  const int per_unit = p.n_qtiles;  // workgroups per unit
  if (!PACKED && !DIRECT && p.by_sweep) {
    kvh = blockIdx.x % p.gn;
    if (!pick_by_sweep(p, blockIdx.x / p.gn, seq, q_lo, L, C, v0)) return;
  } else {
    slice = blockIdx.x / (kXcds * per_unit);
    const int within = blockIdx.x - slice * (kXcds * per_unit);
    const int unit = slice * kXcds + (within % kXcds);
    if (unit >= p.n_units) return;
    const int rank = unit / p.gn;
    kvh = unit - rank * p.gn;
    r = within / kXcds;
    pick_sequence(p, rank, seq, q_lo, L, C);
  }
  // (one value for the workgroup on either way here: the tiles' addresses are scalars)
  seq = __builtin_amdgcn_readfirstlane(seq);
  kvh = __builtin_amdgcn_readfirstlane(kvh);
  L = __builtin_amdgcn_readfirstlane(L);
  C = __builtin_amdgcn_readfirstlane(C);
  const bool causal = p.causal;
  if (L < 0) L = 0;
  if (causal && C > L) C = L;  // under the causal rule a chunk cannot be longer than its context
  // wave blocks per head (a packed mask's lists belong to 128 rows of one head: four blocks, unused ones too)
  const int n_blocks = PACKED ? ((C + 127) >> 7) * kShortWaves : (C + 31) >> 5;
  const int total = n_blocks * p.group;
  // The last blocks (the longest sweeps) first; in the slices that share the CUs with the first ones when
  // the whole grid is resident, last: a CU then holds a long and a short sweep, not two of the same length.
  if (PACKED || DIRECT || !p.by_sweep) v0 = (slice < p.flip_slice ? per_unit - 1 - r : r) * kShortWaves;
  if (v0 >= total) return;

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane((tid / kWave) % kShortWaves);
  const int tg = TG > 1 ? __builtin_amdgcn_readfirstlane(tid / kWave / kShortWaves) : 0;  // tile group
  char *const tiles_k = s_tiles + tg * 2 * NB * TILEB;
  char *const tiles_v = tiles_k + NB * TILEB;
  const int n = lane & 31;  // query column of this lane within the wave's 32-row block
  const int hh = lane >> 5;  // which half of each k-step this lane feeds
  const int v = v0 + wave < total ? v0 + wave : total - 1;
  constexpr bool kByHead = PACKED || DIRECT;  // wave blocks are numbered head by head
  const int head = kByHead ? v / n_blocks : v % p.group;
  const int row0 = (kByHead ? v - head * n_blocks : v / p.group) * 32;
  const bool mine = v0 + wave < total && row0 < C;
  const int h = kvh * p.group + head;
  const int my_q = row0 + n;
  if (L == 0) {  // query rows without any key (not under the causal rule): zero rows
    if (mine && tg == 0 && my_q < C)
#pragma unroll
      for (int c = 0; c < HD / 16; ++c)
        store16(p.out + (query_row(p, q_lo, my_q) * p.out_stride_token + (int64_t)h * HD + (hh * (HD / 16) + c) * 8) * 2,
                Vec16{{0u, 0u, 0u, 0u}});
    return;
  }
  const int P = L - C;  // cached prefix (causal rule only)

  const int qrow = my_q < C ? my_q : C - 1;
  const int limit = causal ? P + qrow : L - 1;  // last key this query row may see
  // Query rows come in whole rows of the head, CPR lanes to a row (a lane's MFMA operands are 16-byte pieces of 32 rows,
  // and loads of those cost a cache line look-up each), are rotated there, and change places through the part
  // of this wave's second tile buffers.
  const int cc = lane % CPR;    // 16-byte chunk of a row this lane moves, here and in the staging below
  const int rsub = lane / CPR;  // row within the rows one load covers
  const int k_lane = n * ROWB + ((hh ^ tile_swizzle_k<CPR>(n)) << 4);  // operand reads of rows stored as K tiles are
  const int my_row = (int)query_row(p, q_lo, qrow);
  Vec16 qf[KS];
  if constexpr (DIRECT) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = load16(p.q + ((int64_t)my_row * p.q_stride_token + (int64_t)h * HD + ks * 16 + hh * 8) * 2);
    if (!PACKED && p.positions != nullptr) {
      const int64_t trig = (int64_t)rope_position(p, my_row) * p.half_hd + hh * 4;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        qf[ks] = rotate_chunk<typename M::E>(qf[ks], p.cos_table + trig + ks * 8, p.sin_table + trig + ks * 8);
    }
  } else {
    int table_row_of_mine = 0;
    if (p.positions != nullptr) table_row_of_mine = rope_position(p, my_row);
    char *const s_q = (wave < 2 ? tiles_k : tiles_v) + (NB - 1) * TILEB + (wave & 1) * (TILEB / 2);
#pragma unroll
    for (int i = 0; i < KS; ++i)
      qf[i] = load16(p.q + ((int64_t)__shfl(my_row, i * WR + rsub, kWave) * p.q_stride_token + (int64_t)h * HD + cc * 8) * 2);
    if (p.positions != nullptr) {
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const int64_t trig = (int64_t)__shfl(table_row_of_mine, i * WR + rsub, kWave) * p.half_hd + cc * 4;
        qf[i] = rotate_chunk<typename M::E>(qf[i], p.cos_table + trig, p.sin_table + trig);
      }
    }
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int r = i * WR + rsub;
      store16(s_q + r * ROWB + ((cc ^ tile_swizzle_k<CPR>(r)) << 4), qf[i]);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = load16(s_q + (k_lane ^ (ks * 32)));
  }

  f32x16_t o[OB];
  float m = kNegInf, l = 0.f;
#pragma unroll
  for (int ob = 0; ob < OB; ++ob)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[ob][i] = 0.f;

  // tiles this wave's rows reach, and the most that any wave of the workgroup does: its last block's
  const int v_last = v0 + kShortWaves < total ? v0 + kShortWaves - 1 : total - 1;
  int last_row = (v_last / p.group) * 32 + 32;  // (a packed mask has its lists instead)
  if (DIRECT) last_row = v0 / n_blocks == v_last / n_blocks ? (v_last % n_blocks) * 32 + 32 : C;
  int kv_end = causal ? P + last_row : L;
  kv_end = kv_end < L ? kv_end : L;
  MaskList list;
  if constexpr (PACKED) list.open(p, seq, h, row0 >> 7, wave);
  const int n_tiles = PACKED ? list.count : __builtin_amdgcn_readfirstlane((kv_end + kBN - 1) / kBN);
  int my_end = causal ? P + row0 + 32 : L;
  my_end = my_end < kv_end ? my_end : kv_end;
  const int my_tiles = mine ? (my_end + kBN - 1) / kBN : 0;

  // ---- tile staging: memory -> LDS (see the long kernel: one table entry and one base address per
  // 16-row group, fixed lane offsets, unconditional loads) -----------------------------------------
  const int64_t head_bytes = (int64_t)kvh * p.stride_head * 2;
  const uint32_t block_bytes = (uint32_t)(p.stride_block * 2);
  const uint32_t token_bytes = (uint32_t)(p.stride_token * 2);
  const int last_phys = (int)p.num_blocks - 1;
  auto block_of = [&](int row) { return (int)__umulhi((uint32_t)row, p.block_magic); };
  const int last_blk = SINGLE ? 0 : block_of(L - 1);
  typedef const __attribute__((address_space(4))) int32_t *TablePtr;  // scalar (SMEM) loads
  const TablePtr table_row = (TablePtr)(unsigned long long)(p.block_tables + (int64_t)seq * p.bt_stride);
  uint32_t src_k[NST], src_v[NST];  // byte offset from the group's first row, less the load's instruction offset
#pragma unroll
  for (int i = 0; i < NST; ++i) {
    const int r = i * WR + rsub;
    src_k[i] = (uint32_t)((int64_t)r * p.stride_token * 2 + (cc ^ tile_swizzle_k<CPR>(r)) * 16) - i * WR * ROWB;
    src_v[i] = (uint32_t)((int64_t)r * p.stride_token * 2 + (cc ^ tile_swizzle_v<CPR>(r)) * 16) - i * WR * ROWB;
  }
  const uint32_t lds_k = (uint32_t)(size_t)(__attribute__((address_space(3))) char *)&s_tiles[0] + (uint32_t)(tg * 2 * NB * TILEB);
  // What round r visits: `tile` (with a packed mask the list's entry, the classes above the tile's number), the
  // table entry of this wave's group and the group's first row within its block.
  struct Stop {
    int32_t tile, ent;
    int rem;
  };
  auto number = [](const Stop &st) { return PACKED ? MaskList::tile(st.tile) : st.tile; };
  auto lookup = [&](int r) {
    Stop st;
    st.tile = PACKED ? list.entry(r) : r < n_tiles ? r : n_tiles - 1;
    const int first = number(st) * kBN + 16 * wave;
    int blk = SINGLE ? 0 : block_of(first);
    st.rem = first - blk * p.block_size;
    if (SINGLE) st.rem = first;
    blk = blk < last_blk ? blk : last_blk;
    st.ent = SINGLE && p.block_tables == nullptr ? seq : table_row[blk];
    return st;
  };
  const uint32_t lds_words =
      (uint32_t)(size_t)(__attribute__((address_space(3))) char *)&s_words[0] + (uint32_t)((tg * kShortWaves + wave) * NB * 256);
  auto fetch = [&](const Stop &st, int buf) {
    int phys = st.ent;
    // A corrupt table entry must not become an out-of-pool address.
    phys = phys < 0 ? 0 : phys;
    phys = phys > last_phys ? last_phys : phys;
    const uint32_t to = __builtin_amdgcn_readfirstlane(lds_k + (uint32_t)(buf * TILEB + 16 * wave * ROWB));
    const uint64_t block = head_bytes + (uint64_t)(uint32_t)phys * block_bytes;
    if (SINGLE) {
#pragma unroll
      for (int pool = 0; pool < 2; ++pool) {
        const char *base = (pool ? p.v_pool : p.k_pool) + block;
#pragma unroll
        for (int i = 0; i < NST; ++i) {
          const int r = i * WR + rsub;
          int row = st.rem + r;
          row = row < L ? row : L - 1;
          const int chunk = cc ^ (pool ? tile_swizzle_v<CPR>(r) : tile_swizzle_k<CPR>(r));
          const char *src = base + (int64_t)row * p.stride_token * 2 + chunk * 16;
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                       :: "s"(to + pool * NB * TILEB + i * WR * ROWB), "v"(src) : "memory", "m0");
        }
      }
    } else {
      const uint64_t group = block + (uint32_t)st.rem * token_bytes;
#pragma unroll
      for (int pool = 0; pool < 2; ++pool) {
        const char *base = (pool ? p.v_pool : p.k_pool) + group;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" :: "s"(to + pool * NB * TILEB) : "memory", "m0");
#pragma unroll
        for (int i = 0; i < NST; ++i)
          asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2"
                       :: "v"(pool ? src_v[i] : src_k[i]), "s"(base), "n"(i * WR * ROWB) : "memory", "m0");
      }
    }
    if constexpr (PACKED) {
      const char *src = reinterpret_cast<const char *>(list.words) + (int64_t)number(st) * 256 + lane * 4;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
                   :: "s"((uint32_t)__builtin_amdgcn_readfirstlane(lds_words + buf * 256)), "v"(src) : "memory", "m0");
    }
  };

  // per-lane LDS offsets of the operand reads (the swizzles seen from the reading side)
  const int vq = (lane & 15) >> 2;
  const int v_lane = (4 * hh + vq) * ROWB + ((tile_swizzle_v<CPR>(vq) >> 2) << 6) + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
  const int mask_from = __builtin_amdgcn_readfirstlane(causal ? (P + row0 + 1) / kBN : L / kBN);

  f32x16_t s[TB];      // S^T of the tile: (token, query n)
  Vec16 pb[kBN / 16];  // its probabilities as MFMA B operands
  auto scores = [&](int buf) {
    const char *sk = tiles_k + buf * TILEB;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[tb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        const Vec16 a = load16(sk + (k_lane ^ (ks * 32)) + tb * 32 * ROWB);
        s[tb] = M::mma(a, qf[ks], s[tb]);
      }
    }
    // operand reads run ahead of the MFMAs that use them (see the long kernel)
    constexpr int kAhead = TB * KS < 6 ? TB * KS : 6;
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
    for (int i = 0; i < TB * KS - kAhead; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
  };
  auto softmax = [&](int tile, int kind, int buf) {
    // s[tb][i] is (token tile*64 + tb*32 + 4*hh + 8*(i/4) + i%4, query n)
    const int tok_base = tile * kBN + 4 * hh;
    if (tile >= mask_from) {  // tiles that touch the causal diagonal (or the context end)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int tok = tok_base + tb * 32 + 8 * (i / 4) + (i & 3);
          s[tb][i] = tok > limit ? kNegInf : s[tb][i];
        }
    }
    if (PACKED && kind == 1) {  // keys the mask hides from this lane's row (beyond the context -inf stays)
      const uint64_t word = s_words[((tg * kShortWaves + wave) * NB + buf) * 32 + n];
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        const uint32_t w = (uint32_t)(word >> (32 * tb)) >> (4 * hh);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const bool hidden = (w & (1u << (8 * (i / 4) + (i & 3)))) == 0;
          s[tb][i] = hidden ? fminf(s[tb][i], kHiddenScore) : s[tb][i];
        }
      }
    }
    float mx = kNegInf;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[tb][i]);
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
    float ps = 0.f;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[tb][i], p.scale_log2e, neg_ms));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[tb][i + 1], p.scale_log2e, neg_ms));
        ps += p0 + p1;
        pb[2 * tb + i / 8].w[(i & 7) / 2] = M::pack2(p0, p1);
      }
    }
    l += ps;
  };
  auto weighted_values = [&](int buf) {
    const char *sv = tiles_v + buf * TILEB;
#pragma unroll
    for (int kk = 0; kk < kBN / 16; ++kk) {
#pragma unroll
      for (int ob = 0; ob < OB; ++ob) {
        const char *at = sv + (v_lane ^ (ob * 64)) + kk * 16 * ROWB;
        const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t *)(at));
        const s16x4_t hi =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t *)(at + 8 * ROWB));
        const s16x8_t both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        o[ob] = M::mma(__builtin_bit_cast(Vec16, both), pb[kk], o[ob]);
      }
    }
    constexpr int kAheadV = 4;
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAheadV, 0);
#pragma unroll
    for (int i = 0; i < OB * (kBN / 16) - kAheadV; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAheadV, 0);
  };

  // ---- sweep: round i is this group's tile i * TG + tg, computed while the next one is on its way ----
  static_assert(NB == 2, "the wait below is for every load in flight");
  const int rounds = (n_tiles + TG - 1) / TG;
  Stop now = lookup(tg);
  fetch(now, 0);
  Stop next = lookup(TG + tg);
  for (int i = 0; i < rounds; ++i) {
    const int k = i * TG + tg;
    const int buf = i & 1;
    const int tile = number(now);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's groups of the round's tile
    // rows of a V tile past the context become zeros: their probabilities are zeros, but 0 x NaN is not,
    // and unused pool slots may hold anything (only a sweep's last tile can reach past the context)
    if (tile * kBN + 16 * wave + 16 > L) {
      char *at = tiles_v + buf * TILEB + 16 * wave * ROWB + lane * 16;
      const int row = tile * kBN + 16 * wave + rsub;
#pragma unroll
      for (int j = 0; j < NST; ++j)
        if (row + j * WR >= L) store16(at + j * WR * ROWB, Vec16{{0u, 0u, 0u, 0u}});
    }
    __syncthreads();  // the round's tiles are whole, and nobody reads the buffer of the round before any more
    fetch(next, buf ^ 1);  // (past the sweep the last tile is fetched again: nobody reads it)
    const int kind = PACKED ? MaskList::kind(now.tile, wave) : 2;
    now = next;
    next = lookup(k + 2 * TG);
    if (PACKED ? (k < n_tiles && mine && kind != 0) : k < my_tiles) {
      scores(buf);
      softmax(tile, kind, buf);
      weighted_values(buf);
    }
  }
  // every load this wave issued must have landed before its LDS is given up
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- the second group's sums -----------------------------------------------------------
  if constexpr (TG > 1) {
    static_assert(TG == 2, "one hand-over");
    float *slab = reinterpret_cast<float *>(s_tiles) + wave * (OB * 16 + 2) * kWave + lane;
    __syncthreads();
    if (tg == 1) {
#pragma unroll
      for (int ob = 0; ob < OB; ++ob)
#pragma unroll
        for (int i = 0; i < 16; ++i) slab[(ob * 16 + i) * kWave] = o[ob][i];
      slab[OB * 16 * kWave] = m;
      slab[(OB * 16 + 1) * kWave] = l;
    }
    __syncthreads();
    if (tg == 1) return;
    const float m1 = slab[OB * 16 * kWave], l1 = slab[(OB * 16 + 1) * kWave];
    const float m_new = fmaxf(m, m1);
    const float w0 = m == kNegInf ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
    const float w1 = m1 == kNegInf ? 0.f : __builtin_amdgcn_exp2f(m1 - m_new);
    l = l * w0 + l1 * w1;
#pragma unroll
    for (int ob = 0; ob < OB; ++ob)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[ob][i] = o[ob][i] * w0 + slab[(ob * 16 + i) * kWave] * w1;
  }

  // ---- normalise and store -------------------------------------------------------
  float l_a, l_b;
  both_halves(l, l_a, l_b);
  const float lt = l_a + l_b;
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  if constexpr (DIRECT) {
    if (mine && my_q < C) {
      // (a packed mask comes with equal sequences, whose rows need no register until here)
      char *const orow = p.out + ((PACKED ? q_lo + my_q : my_row) * p.out_stride_token + (int64_t)h * HD + 4 * hh) * 2;
#pragma unroll
      for (int ob = 0; ob < OB; ++ob) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint2 w;
          w.x = M::pack2(o[ob][4 * j] * inv, o[ob][4 * j + 1] * inv);
          w.y = M::pack2(o[ob][4 * j + 2] * inv, o[ob][4 * j + 3] * inv);
          *reinterpret_cast<uint2 *>(orow + (ob * 32 + 8 * j) * 2) = w;
        }
      }
    }
    return;
  }
  // Out in whole rows of the head again, through LDS: the tiles are done with (with two tile groups the first group's
  // wave takes the slab it has just read).
  if constexpr (TG == 1) __syncthreads();
  char *const s_o = TG == 1 ? s_tiles + wave * 32 * ROWB : s_tiles + wave * (OB * 16 + 2) * kWave * 4;
#pragma unroll
  for (int ob = 0; ob < OB; ++ob) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint2 w;
      w.x = M::pack2(o[ob][4 * j] * inv, o[ob][4 * j + 1] * inv);
      w.y = M::pack2(o[ob][4 * j + 2] * inv, o[ob][4 * j + 3] * inv);
      *reinterpret_cast<uint2 *>(s_o + n * ROWB + (((ob * 4 + j) ^ tile_swizzle_k<CPR>(n)) << 4) + hh * 8) = w;
    }
  }
#pragma unroll
  for (int i = 0; i < KS; ++i) {
    const int r = i * WR + rsub;
    const int64_t row = PACKED ? q_lo + row0 + r : __shfl(my_row, r, kWave);
    const int64_t to = row * p.out_stride_token + (int64_t)h * HD + cc * 8;
    const Vec16 v = load16(s_o + r * ROWB + ((cc ^ tile_swizzle_k<CPR>(r)) << 4));
    if (mine && row0 + r < C) store16(p.out + to * 2, v);
  }
}

template <class M, bool SINGLE, int TG, bool PACKED, bool DIRECT>
int launch_short_hd(const PrefillKP &kp, int hd, unsigned wgs, hipStream_t stream) {
  const dim3 grid(wgs), block(TG * kShortWaves * kWave);
  switch (hd) {
    case 32:
      hipLaunchKernelGGL((paged_prefill_short_kernel<M, 32, SINGLE, TG, PACKED, DIRECT>), grid, block, 0, stream, kp);
      break;
    case 64:
      hipLaunchKernelGGL((paged_prefill_short_kernel<M, 64, SINGLE, TG, PACKED, DIRECT>), grid, block, 0, stream, kp);
      break;
    case 128:
      hipLaunchKernelGGL((paged_prefill_short_kernel<M, 128, SINGLE, TG, PACKED, DIRECT>), grid, block, 0, stream, kp);
      break;
    default:
      return IC_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

template <class M, bool DIRECT>
int launch_short_type(const PrefillKP &kp, const PrefillArgs &a, unsigned wgs, bool split, hipStream_t stream) {
  if (a.mask_bits != nullptr)
    return split ? launch_short_hd<M, true, 2, true, DIRECT>(kp, a.hd, wgs, stream)
                 : launch_short_hd<M, true, 1, true, DIRECT>(kp, a.hd, wgs, stream);
  if (a.block_tables == nullptr || a.block_table_stride == 1)
    return split ? launch_short_hd<M, true, 2, false, DIRECT>(kp, a.hd, wgs, stream)
                 : launch_short_hd<M, true, 1, false, DIRECT>(kp, a.hd, wgs, stream);
  return split ? launch_short_hd<M, false, 2, false, DIRECT>(kp, a.hd, wgs, stream)
               : launch_short_hd<M, false, 1, false, DIRECT>(kp, a.hd, wgs, stream);
}

}  // namespace

// Which kernel a 16-bit call without a mask takes.  The host knows the longest chunk and, from the
// block table, a bound on the contexts.  Times in us, 16 sequences, 32 query heads, head dim 128, this
// kernel / the long one, by chunk length and cached prefix:
//                     32 KV heads                            8 KV heads
//   prefix      0       1 024     2 048      4 096       0      1 024     2 048      4 096
//   chunk 128  18 / 25   70 / 79  119 / 130  220 / 228   15 / 22  46 / 63   78 / 99   160 / 182
//         256  35 / 43  118 / 114 193 / 177  347 / 311   31 / 41  90 / 97  153 / 153  299 / 270
//         384  52 / 71  168 / 178 270 / 290  484 / 507   49 / 66 136 / 161 226 / 251  432 / 450
//         512  83 / 97  227 / 219 359 / 334  636 / 578   76 / 91 197 / 199 336 / 312  595 / 532
//       1 024 239 / 268 485 / 485 740 / 710 1246 / 1165 217 / 265 450 / 477 698 / 689 1180 / 1118
// The long kernel needs its 256 rows filled and long full sweeps (a prefix at least as long as the
// chunk), where staging a tile once per 256 rows instead of 128 pays; sooner without grouped queries,
// whose K/V the caches do not serve to several heads.  A grid that leaves the CUs one workgroup each is this
// kernel's (with two tile groups, below: 2 sequences, chunks of 128 behind 4 096: 66 / 78 us, grouped 64 / 78)
// unless it streams many ungrouped K/V rows, for which the long kernel keeps more bytes on their way (4
// sequences behind 4 096 / 8 192: 84 / 81 and 164 / 149 us).  At head dim 64 and 32 (half the staged bytes per
// row, four workgroups per CU) this one is within 4 % at worst (512 behind 4 096: 354 / 351) and up to a third
// faster.
namespace {
int64_t short_workgroups_per_unit(const PrefillArgs &a) {
  const int64_t per_head = a.mask_bits ? (int64_t)((a.max_chunk_len + 127) / 128) * kShortWaves : (a.max_chunk_len + 31) / 32;
  const int64_t blocks = per_head * (a.hn / a.gn);
  return (blocks + kShortWaves - 1) / kShortWaves;
}
int64_t context_bound(const PrefillArgs &a) {
  return a.context_lens == nullptr ? a.uniform_context : a.block_table_stride * (int64_t)a.pool.block_size;
}
}  // namespace

bool prefill_takes_short(const PrefillArgs &a) {
  if (a.hd < 128) return true;
  const int64_t ctx = context_bound(a);
  const int64_t wgs = short_workgroups_per_unit(a) * a.n_seqs * a.gn;
  if (wgs <= device_cu_count()) return a.hn > a.gn || wgs * ctx < 512 * 1024;
  const int tiles = (a.max_chunk_len + 255) / 256;
  const bool filled = (int64_t)a.max_chunk_len * 8 >= (int64_t)tiles * 256 * 7;
  return !(filled && ctx >= 2 * (int64_t)a.max_chunk_len && ctx >= (a.hn > a.gn ? 2200 : 1250));
}

namespace {
// A few query rows to a chunk, which gain nothing from being moved as whole rows (figures below).
bool few_rows(const PrefillArgs &a) { return a.max_chunk_len <= (a.hd == 128 && a.hn > a.gn ? 4 : 8); }

// Whether query rows and outputs move as the MFMA lays them out, without the exchange in LDS: that exchange costs a
// workgroup half a microsecond of latency and saves its CU's cache look-ups, so it loses where the launch is over in a few
// tiles or leaves the CUs a workgroup or two.  Rotary tables are read by whole rows too, which gains from a few rows on:
// chunks of 2 / 4 / 8 / 16 / 32 rows (1-42 sequences, nothing to 2 000 cached tokens, append and attention) take 4.5 / 3 / 2 /
// -1.5 / -9 % more by whole rows at head dim 128, 2 / 1.5 / -1 / -7 / -14 % with grouped heads (42 x 2, 8 / 8 heads of 128:
// 15.7 / 14.4 us), 4 / 3 / 2 / 0 / -6 % at 64.  As few rows without rotary gain alike (64 x 3, 16 / 4 heads of 128: 13.8 / 13.2).
// More rows without it, us by whole rows / directly (calls without a cache):
//   sequences x tokens            1 x 20       18 x 70       3 x 300       4 x 500       60 x 100      30 x 130      2 x 1 024
//   12 / 12 heads of 64, causal   4.9 / 4.3    6.6 / 5.7     9.3 / 8.2    13.0 / 11.7   11.5 / 10.9   10.1 / 10.1   16.4 / 16.4
//                  all keys       5.0 / 4.3    6.5 / 6.0     9.5 / 9.0    13.2 / 12.5   11.6 / 12.1   11.7 / 12.9   16.5 / 16.4
//             packed documents    5.7 / 4.8    7.4 / 6.6     9.9 / 9.0    11.7 / 10.7   12.9 / 12.6   11.0 / 11.0   12.8 / 13.0
//   16 / 16 of 128, causal        5.9 / 5.4   10.0 / 9.3    11.1 / 10.5   16.7 / 16.1   24.6 / 24.9   21.4 / 22.6   23.2 / 24.0
//                  all keys       5.8 / 5.1    9.8 / 10.5   11.6 / 12.3   17.5 / 18.1   25.2 / 28.3   23.5 / 27.9   24.3 / 26.2
//             packed documents    6.3 / 5.6   10.7 / 9.9    11.4 / 11.2   14.7 / 14.5   26.1 / 26.9   22.8 / 24.1   17.4 / 18.9
//   80 x 129, 12 / 12 of 64, causal (1 920 workgroups): 18.8 / 20.8; packed, 60 x 20, 64 / 8 of 128: 44.1 / 38.1.
// (A packed mask at head dim 64 loses where two tile groups share the tiles, 2 x 1 024 tokens of 16 heads 13.0 / 13.3, 1 x 700 of 12
// 10.0 / 10.3, and gains in the larger grids without, 3 x 1 500 of 12 heads 21.2 / 20.2.)
// Grouped heads put one row block of several heads into a workgroup, which reaches equally far, where this numbers head
// by head: only in grids of a workgroup to a CU (8 / 1 of 64, causal, 8 x 70 6.1 / 5.6, 3 x 300 9.5 / 8.7, 2 x 1 024 23 % faster
// by whole rows; at head dim 128, 28 / 4, causal, 8 x 70 8.1 / 7.7, 1 x 20 9 % faster by whole rows).
bool prefill_rows_direct(const PrefillArgs &a, int64_t wgs, bool two_groups) {
  const int64_t cus = device_cu_count(), ctx = context_bound(a);
  const bool packed = a.mask_bits != nullptr;
  if (!packed && few_rows(a)) return true;
  if (a.positions != nullptr) return false;
  if (a.hn > a.gn && !packed) return wgs <= cus && (a.hd < 128 ? ctx <= 512 : a.causal && ctx > 64 && ctx <= 128);
  if (a.hd < 128) return packed ? !two_groups : ctx <= 64 || wgs <= (a.causal ? 4 : 1) * cus;
  if (ctx <= 64) return true;
  if (packed) return a.max_chunk_len <= 128 && wgs <= 5 * cus;
  return a.causal ? ctx <= 320 && 2 * wgs <= 5 * cus : ctx <= 128 && wgs <= cus;
}
}  // namespace

int launch_paged_prefill_short(PrefillKP kp, const PrefillArgs &a, hipStream_t stream) {
  const int64_t per_unit = short_workgroups_per_unit(a);
  const int64_t slices = (kp.n_units + kXcds - 1) / kXcds;
  int64_t wgs = slices * kXcds * per_unit;
  // Chunks that lie in padded rows are of unequal length.  Numbered unit by unit, an XCD gets `slices` units and is
  // uneven against the others where they, or a single one, are more workgroups than its CUs hold at once; where they
  // are not, everything is resident anyway and the search in each workgroup (1-1.5 us) is lost.  us by sweep / by unit (append
  // and attention), workgroups of a unit x units of an XCD of the padded chunks, nothing cached and up to 1 024, 8 192 tokens:
  //   28 / 4 heads of 128, 9 of 3-701 rows     37 x 5     37.6 / 39.7    61.2 / 71.0
  //                        9 of 100-500        27 x 5     31.2 / 32.4    52.5 / 58.7
  //                       16 of 10-200         13 x 8     21.2 / 22.7    39.5 / 40.7   166.9 / 175.9
  //                        9 of 3-60            4 x 5     10.5 / 10.0    24.5 / 22.4   111.5 / 108.3
  //    8 / 1 of 128,       9 of 3-701          42 x 2     25.5 / 26.1    35.1 / 39.0   120.3 / 146.8
  //                       32 of 3-60            4 x 4     12.2 / 11.7    29.2 / 25.6
  //   32 / 32 of 128,     32 of 100-500         4 x 128  168.3 / 193.7
  //                        2 of 100-500         4 x 8     22.3 / 21.6    33.1 / 31.7
  //   16 / 4 of 64,        9 of 3-701          21 x 5     25.8 / 24.3    38.6 / 37.3
  //                       32 of 3-701          22 x 16    47.8 / 51.4    75.4 / 80.2
  //   16 / 16 of 64,      32 of 100-500         4 x 64    51.6 / 53.9    76.2 / 80.3
  //                        9 of 100-500         4 x 18    25.3 / 24.3    37.6 / 36.5
  // (954 sizes measured, 2-60 sequences, 1-32 KV heads: by this line 2.2 % less time than by unit throughout, 2.9 % less
  // than by sweep throughout, 0.5 % more than the better of the two.)
  const int64_t xcd_cus = device_cu_count() / kXcds;
  // (Few rows to a chunk: directly, below, which gains more: 26 chunks of 3-8, 32 / 32 heads of 128: 39.3 / 37.3.)
  kp.by_sweep = a.rows != nullptr && a.mask_bits == nullptr && a.n_seqs <= kWave && !few_rows(a) &&
                (per_unit > xcd_cus || slices * per_unit > xcd_cus * (a.hd == 128 ? 2 : 4));
  if (kp.by_sweep) {  // (at most so many workgroups, a sequence's last one and row block not full)
    const int64_t blocks = a.n_rows / 32 + a.n_seqs;
    wgs = a.gn * ((blocks * kp.group + kShortWaves - 1) / kShortWaves + a.n_seqs);
  }
  if (wgs > 0x7fffffff) return IC_ERR_UNSUPPORTED;
  kp.n_qtiles = (int)per_unit;
  const int cus = device_cu_count();
  kp.flip_slice = wgs > cus && wgs <= 2 * cus ? (int)(slices + 1) / 2 : 0x7fffffff;
  // A grid that leaves the CUs one workgroup each: two groups of waves take the tiles in turn.  2 sequences,
  // 32 heads of 128, chunks of 128 behind 512 / 1 024 / 4 096 cached tokens: 16.8 / 28.2 / 86.3 us with one
  // group, 16.6 / 24.9 / 66.0 with two; behind nothing 7.8 / 10.0 (the hand-over), hence the second condition.
  // At head dim 64 two such workgroups share a CU: 16 sequences, chunks of 128 behind 512 / 2 048 / 4 096:
  // 22.6 / 69.6 / 137 with one group, 24.4 / 65.4 / 128 with two.
  const int64_t ctx = context_bound(a);
  const bool split = (wgs <= cus && ctx > 512) || (a.hd < 128 && wgs <= 2 * cus && ctx >= 2048);
  const bool bf16 = a.dtype == IC_DTYPE_BF16;
  if (!kp.by_sweep && prefill_rows_direct(a, per_unit * kp.n_units, split))
    return bf16 ? launch_short_type<MmaBf16, true>(kp, a, (unsigned)wgs, split, stream)
                : launch_short_type<MmaF16, true>(kp, a, (unsigned)wgs, split, stream);
  return bf16 ? launch_short_type<MmaBf16, false>(kp, a, (unsigned)wgs, split, stream)
              : launch_short_type<MmaF16, false>(kp, a, (unsigned)wgs, split, stream);
}

}  // namespace prefill
}  // namespace ic
