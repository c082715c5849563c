// How the append kernels (kv_append.hip, rope_kv_append.hip) lay token rows over
// workgroups of kAppendThreads lanes, one 16-byte chunk of a row to a lane.
#pragma once

#include "ic_device.h"
#include "ic_internal.h"

namespace ic {

constexpr int kAppendThreads = 256;
constexpr int kAppendThreadsShift = 8;

// Lanes a row takes in a workgroup, as a shift: a row that fills less than a workgroup shares it.  A few KV
// heads are a wave's worth of chunks (4 heads of 128 in 16 bits: 64), and with a workgroup to a row the launch
// is bound by how fast workgroups start and three quarters of their lanes do nothing.
// 9 chunks padded to 701 tokens, 4 KV heads of 128, rotary, query rotated elsewhere: 4 us (the layer call
// 56.2 -> 51.9); 8 192 tokens of 32 heads, whose rows fill their workgroups, as before.
inline int append_row_shift(int chunks) {
  int shift = 0;
  while (shift < kAppendThreadsShift && (1 << shift) < chunks) ++shift;
  return shift;
}

// Token (from the slice's first) and chunk of this lane.  A row that fills the workgroup is the same for all
// its lanes (WIDE: its slot and the division by the block size stay scalar).
template <bool WIDE>
__device__ __forceinline__ int64_t append_token(int row_shift) {
  if (WIDE) return blockIdx.y;
  return ((int64_t)blockIdx.y << (kAppendThreadsShift - row_shift)) + (threadIdx.x >> row_shift);
}
template <bool WIDE>
__device__ __forceinline__ int append_chunk(int row_shift) {
  return blockIdx.x * kAppendThreads + (WIDE ? threadIdx.x : threadIdx.x & ((1 << row_shift) - 1));
}

// Block of a slot in [0, num_slots): where a lane's slots differ, a 64-bit division on the vector unit is some
// hundred instructions.
template <bool WIDE>
__device__ __forceinline__ int64_t slot_block(int64_t slot, int block_size, int64_t num_slots) {
  if (WIDE || (num_slots >> 32) != 0) return slot / block_size;
  return (uint32_t)slot / (uint32_t)block_size;
}

// Zeroes the rows of a padded output that no chunk holds, ahead of the attention launch that writes the others.
// Bound by the bytes written.  Row r of sequence i is known to be listed when entry bounds[i] + r names it (chunks
// at the start of their rows, what PagedKVCache lays out); a row listed elsewhere is zeroed and written again,
// which is why this comes before the attention kernel: inside it it would race with that write.  It is a part of the
// append's launch (9 prompts padded to 701 rows of 28 heads of 128: one launch of 7 us instead of 7 + 6).
__device__ __forceinline__ void zero_unlisted_rows(const ZeroRows &z, int64_t group, int64_t groups) {
  for (int64_t row = group; row < z.total; row += groups) {
    const int seq = (int)(row / z.row_pitch);
    const int64_t at = z.bounds[seq] + (row - (int64_t)seq * z.row_pitch);
    if (at >= 0 && at < z.bounds[seq + 1] && at < z.n_rows && z.rows[at] == row) continue;
    for (int c = threadIdx.x; c < z.chunks; c += kAppendThreads)
      store16(z.out + row * z.stride_bytes + (int64_t)c * 16, Vec16{{0u, 0u, 0u, 0u}});
  }
}

// The z slices of an append's grid behind its own parts are that, if there is anything to zero: as many as bring the
// workgroups that the rows alone would get (zero_slices; a narrow model's append has a handful, and rows zeroed one after
// the other by those cost more than the launch that is saved: 2 prompts of 3-60 tokens, 8 query heads on one KV head of
// 64: 17.2 us for the layer call, 8.5 so, 10.4 with a launch of its own).
__device__ __forceinline__ bool zero_part(const ZeroRows &z, unsigned parts) {
  if (blockIdx.z < parts) return false;
  const int64_t slice = (int64_t)gridDim.y * gridDim.x;
  zero_unlisted_rows(z, (blockIdx.z - parts) * slice + (int64_t)blockIdx.y * gridDim.x + blockIdx.x,
                     (gridDim.z - parts) * slice);
  return true;
}

// (host) Workgroups for `total` rows, and the slices of an append's grid that hold them.
inline int64_t zero_workgroups(int64_t total) {
  const int64_t most = (int64_t)device_cu_count() * 8;
  return total < most ? total : most;
}
inline unsigned zero_slices(const ZeroRows &z, const dim3 &grid) {
  const int64_t slice = (int64_t)grid.y * grid.x;
  return (unsigned)((zero_workgroups(z.total) + slice - 1) / slice);
}

}  // namespace ic
