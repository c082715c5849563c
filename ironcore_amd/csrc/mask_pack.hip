// Packs a general attention mask for the prefill kernels.
//
// The reference takes any mask broadcastable to [b, hn, sq, sk] (attention.py:
// 115-117) and adds its fill value to every score.  Read byte by byte inside the
// attention kernel a mask costs 32 loads per lane and K/V tile, and the sweep
// walks every tile whatever the mask hides.  This kernel reads the bytes once
// (for all heads that share them, and for all layers of a forward pass: the
// layer keeps the result with the mask) and leaves
//
//   bits   one 64-bit word per (query row, 64-key tile), as [32-row group][tile][row]
//          so that a wave of the attention kernel fetches its tile's words as 256
//          consecutive bytes;
//   lists  per 128-row query tile the K/V tiles that any of its rows sees, each
//          with the class of the four 32-row groups: 0 nothing visible, 1 mixed,
//          2 everything visible.  A row that sees no key at all averages V over
//          the whole context (finite fill value), so a query tile with such a row
//          lists every tile and the row's group skips none;
//   flags  whether the mask hides nothing, and whether it is the causal pattern.
//
// One workgroup per (query tile, head, sequence); 16 waves: wave w packs 32-row
// group w % 4 of tiles w / 4, w / 4 + 4, ...  A lane turns 32 bytes of a row into
// 32 bits.  Bound by the latency of a tile's loads.  The layer's first call on a
// new mask of 2 x 1 024 x 1 024 bytes (16 heads of 64, synchronisation and attention
// included) takes 103 us; with a dozen elementwise passes to classify and copy
// the mask and the byte path behind them it took 344.
#include "ic_device.h"
#include "ic_internal.h"
#include "../../include/ironcore_paged.h"

namespace ic {

namespace {

constexpr int kPackThreads = 1024;
constexpr int kPackMaxTiles = 8192;  // class bytes of a query tile in LDS: 4 per tile

struct PackKP {
  const uint8_t *mask;
  int64_t stride_seq, stride_head, stride_row;
  int rows, keys, n_tiles, n_qtiles;
  uint64_t *bits;
  int32_t *lists;
  int32_t *flags;
};

// Bit k of the result: byte k of the four in w is not zero.
__device__ __forceinline__ uint32_t nonzero4(uint32_t w) {
  const uint32_t t = (((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) & 0x80808080u;
  return ((t >> 7) * 0x10204080u) >> 28;  // bits 0, 8, 16, 24 gathered into 28 .. 31, in order
}

// First n (clamped to 0 .. 64) bits set.
__device__ __forceinline__ uint64_t low_bits(int n) { return n <= 0 ? 0 : n >= 64 ? ~0ull : (1ull << n) - 1; }

__global__ __launch_bounds__(kPackThreads) void mask_pack_kernel(const PackKP p) {
  extern __shared__ uint8_t s_class[];  // [tile][4]
  __shared__ uint32_t s_seen[4];        // per row group: rows that see a key
  __shared__ int s_flags;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int group = wave & 3;
  const int qt = blockIdx.x;
  const int64_t plane = (int64_t)blockIdx.z * gridDim.y + blockIdx.y;
  if (threadIdx.x < 4) s_seen[threadIdx.x] = 0;
  if (threadIdx.x == 0) s_flags = 3;
  __syncthreads();
  const int row_in_group = lane >> 1, half = lane & 1;
  const int row = qt * 128 + group * 32 + row_in_group;
  const bool exists = row < p.rows;
  const uint8_t *bytes = p.mask + blockIdx.z * p.stride_seq + blockIdx.y * p.stride_head +
                         (int64_t)(exists ? row : p.rows - 1) * p.stride_row;
  uint64_t *bits = p.bits + ((plane * p.n_qtiles + qt) * 4 + group) * p.n_tiles * 32 + row_in_group;
  bool seen = false;
  int flags = 3;  // bit 0: hides nothing so far, bit 1: causal so far
  for (int t = wave >> 2; t < p.n_tiles; t += 4) {
    const int j0 = t * 64 + half * 32;
    uint32_t mine = 0;
    if (j0 + 32 <= p.keys) {
      uint32_t w[8];
      __builtin_memcpy(w, bytes + j0, 32);
#pragma unroll
      for (int k = 0; k < 8; ++k) mine |= nonzero4(w[k]) << (4 * k);
    } else {
      for (int k = 0; j0 + k < p.keys; ++k) mine |= (bytes[j0 + k] != 0 ? 1u : 0u) << k;
    }
    const uint32_t other = __shfl_xor(mine, 1, kWave);
    uint64_t word = half == 0 ? (uint64_t)mine | ((uint64_t)other << 32) : (uint64_t)other | ((uint64_t)mine << 32);
    if (!exists) word = 0;
    if (half == 0) bits[(int64_t)t * 32] = word;
    seen |= word != 0;
    const uint64_t in_range = low_bits(p.keys - t * 64);
    if (exists && word != in_range) flags &= ~1;
    if (exists && word != (in_range & low_bits(p.keys - p.rows + row + 1 - t * 64))) flags &= ~2;
    const bool none = __all(word == 0);
    const bool full = __all(!exists || word == ~0ull);
    if (lane == 0) s_class[t * 4 + group] = none ? 0 : full ? 2 : 1;
  }
  // (even lanes speak for their row)
  const uint64_t saw = __ballot(seen && half == 0);
  if (lane == 0) {
    uint32_t rows = 0;
    for (int r = 0; r < 32; ++r) rows |= (uint32_t)((saw >> (2 * r)) & 1) << r;
    atomicOr(&s_seen[group], rows);
  }
  if (!__all((flags & 1) != 0) && lane == 0) atomicAnd(&s_flags, ~1);
  if (!__all((flags & 2) != 0) && lane == 0) atomicAnd(&s_flags, ~2);
  __syncthreads();
  if (threadIdx.x == 0) {
    if (!(s_flags & 1)) atomicAnd(&p.flags[0], 0);
    if (!(s_flags & 2)) atomicAnd(&p.flags[1], 0);
  }
  if (wave != 0) return;
  // ---- the query tile's list, 64 tiles at a time ------------------------------------------
  int blind = 0;  // bit g: a row of group g sees nothing
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int n = p.rows - (qt * 128 + g * 32);
    const uint32_t want = (uint32_t)low_bits(n < 32 ? n : 32);
    if ((s_seen[g] & want) != want) blind |= 1 << g;
  }
  int32_t *list = p.lists + (plane * p.n_qtiles + qt) * (p.n_tiles + 1);
  int count = 0;
  for (int base = 0; base < p.n_tiles; base += kWave) {
    const int t = base + lane;
    int entry = 0;
    if (t < p.n_tiles) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        int c = s_class[t * 4 + g];
        if (c == 0 && ((blind >> g) & 1)) c = 1;
        entry |= c << (16 + 2 * g);
      }
    }
    const bool listed = t < p.n_tiles && (entry != 0 || blind != 0);
    const uint64_t hit = __ballot(listed);
    if (listed) list[1 + count + __builtin_popcountll(hit & low_bits(lane))] = entry | t;
    count += __builtin_popcountll(hit);
  }
  if (lane == 0) list[0] = count;
}

}  // namespace

int launch_mask_pack(const uint8_t *mask, int64_t stride_seq, int64_t stride_head, int64_t stride_row, int n_seqs,
                     int heads, int rows, int keys, uint64_t *bits, int32_t *lists, int32_t *flags,
                     hipStream_t stream) {
  PackKP p;
  p.mask = mask;
  p.stride_seq = stride_seq;
  p.stride_head = stride_head;
  p.stride_row = stride_row;
  p.rows = rows;
  p.keys = keys;
  p.n_tiles = (keys + 63) / 64;
  p.n_qtiles = (rows + 127) / 128;
  p.bits = bits;
  p.lists = lists;
  p.flags = flags;
  if (p.n_tiles > kPackMaxTiles || heads > 65535 || n_seqs > 65535) return IC_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(mask_pack_kernel, dim3(p.n_qtiles, heads, n_seqs), dim3(kPackThreads), (size_t)p.n_tiles * 4, stream,
                     p);
  return hipGetLastError() == hipSuccess ? IC_OK : IC_ERR_LAUNCH;
}

}  // namespace ic
