"""Block KV cache: pools, block allocator with prefix sharing, batch metadata.

The reference has no KV cache (its only generation loop recomputes the whole
sequence every step, examples/generate_text.py:24-40), so this interface is
defined here.  One ``PagedKVCache`` serves all layers of a model:

* per layer a K pool and a V pool ``[num_blocks, gn, block_size, hd]``
  (native layout of the kernels: one (block, KV head) tile is contiguous);
* one block table per sequence, shared by all layers (layer ``l`` of a
  sequence uses the same block ids in layer ``l``'s pools);
* a host-side allocator with reference counts, so sequences forked from a
  common prompt (GRPO groups) alias the prompt's full blocks and copy only the
  partly filled last block.

Everything the kernels need per step comes from :meth:`PagedKVCache.prepare`,
which advances the sequences by the step's new tokens and returns a
``PagedAttentionMetadata`` (block tables, context lengths, slot mapping).  The
allocator state lives on the host; ``prepare`` uploads small int tensors and
never reads anything back from the GPU.
"""
from __future__ import annotations

from dataclasses import dataclass, field
from operator import index
from typing import Iterable, Sequence

import numpy as np
import torch

from .layers.attention import PagedAttentionMetadata


class OutOfBlocks(RuntimeError):
    """The pool has no free block left."""


class BlockAllocator:
    """Free list + reference counts over ``num_blocks`` pool blocks."""

    def __init__(self, num_blocks: int):
        self.num_blocks = num_blocks
        self._free = list(range(num_blocks - 1, -1, -1))
        self._refs = [0] * num_blocks

    @property
    def num_free(self) -> int:
        return len(self._free)

    def allocate(self) -> int:
        if not self._free:
            raise OutOfBlocks(f"all {self.num_blocks} KV blocks are in use")
        blk = self._free.pop()
        self._refs[blk] = 1
        return blk

    def share(self, blk: int) -> int:
        if self._refs[blk] <= 0:
            raise ValueError(f"block {blk} is not allocated")
        self._refs[blk] += 1
        return blk

    def release(self, blk: int) -> None:
        if self._refs[blk] <= 0:
            raise ValueError(f"block {blk} is not allocated")
        self._refs[blk] -= 1
        if self._refs[blk] == 0:
            self._free.append(blk)

    def ref_count(self, blk: int) -> int:
        return self._refs[blk]


@dataclass
class _Sequence:
    blocks: list = field(default_factory=list)
    length: int = 0


class PagedKVCache:
    """Pools for ``num_layers`` layers plus the sequences that live in them."""

    def __init__(self, num_layers: int, num_blocks: int, block_size: int, num_kv_heads: int,
                 head_dim: int, dtype: torch.dtype, device):
        if block_size % 16 != 0:
            raise ValueError("block_size must be a multiple of 16 (the kernels walk 16-token tiles)")
        self.num_layers = num_layers
        self.num_blocks = num_blocks
        self.block_size = block_size
        shape = (num_layers, num_blocks, num_kv_heads, block_size, head_dim)
        self.k_pools = torch.zeros(shape, dtype=dtype, device=torch.device(device))
        self.device = self.k_pools.device    # with its index, whatever the spelling
        self.v_pools = torch.zeros(shape, dtype=dtype, device=self.device)
        self.allocator = BlockAllocator(num_blocks)
        self._seqs: dict[int, _Sequence] = {}
        self._next_id = 0

    # ---- pools -----------------------------------------------------------------
    def layer(self, index: int):
        """(k_pool, v_pool) of one layer, the ``kv_cache`` argument of
        ``Attention.forward``."""
        return self.k_pools[index], self.v_pools[index]

    # ---- sequences ---------------------------------------------------------------
    def add_sequence(self) -> int:
        sid = self._next_id
        self._next_id += 1
        self._seqs[sid] = _Sequence()
        return sid

    def length(self, sid: int) -> int:
        return self._seqs[sid].length

    def blocks(self, sid: int) -> list:
        return list(self._seqs[sid].blocks)

    def free_sequence(self, sid: int) -> None:
        for blk in self._seqs.pop(sid).blocks:
            self.allocator.release(blk)

    def fork(self, sid: int) -> int:
        """New sequence with the same content: full blocks are aliased
        (reference count up), a partly filled last block is copied so that the
        two sequences can append independently."""
        src = self._seqs[sid]
        if src.length % self.block_size and self.allocator.num_free < 1:
            raise OutOfBlocks("no free KV block for the copy of the partly filled block")
        child = _Sequence(length=src.length)
        full = src.length // self.block_size
        for blk in src.blocks[:full]:
            child.blocks.append(self.allocator.share(blk))
        if src.length % self.block_size:
            new = self.allocator.allocate()
            old = src.blocks[full]
            self.k_pools[:, new].copy_(self.k_pools[:, old])
            self.v_pools[:, new].copy_(self.v_pools[:, old])
            child.blocks.append(new)
        cid = self._next_id
        self._next_id += 1
        self._seqs[cid] = child
        return cid

    def _blocks_needed(self, seq: _Sequence, new_tokens: int) -> int:
        """Blocks the allocator must still give for ``new_tokens`` more tokens:
        new ones past the blocks the sequence holds, plus the private copy of a
        shared block that the next token would be written into."""
        if new_tokens <= 0:
            return 0
        bs = self.block_size
        need = max((seq.length + new_tokens + bs - 1) // bs - len(seq.blocks), 0)
        idx = seq.length // bs
        if idx < len(seq.blocks) and self.allocator.ref_count(seq.blocks[idx]) > 1:
            need += 1
        return need

    def _slot_for_append(self, seq: _Sequence) -> int:
        """Slot of the next token; allocates a block at block boundaries and
        un-shares an aliased block before it is written (copy on write)."""
        bs = self.block_size
        idx, off = divmod(seq.length, bs)
        if idx == len(seq.blocks):
            seq.blocks.append(self.allocator.allocate())
        blk = seq.blocks[idx]
        if self.allocator.ref_count(blk) > 1:
            new = self.allocator.allocate()
            self.k_pools[:, new].copy_(self.k_pools[:, blk])
            self.v_pools[:, new].copy_(self.v_pools[:, blk])
            self.allocator.release(blk)
            seq.blocks[idx] = blk = new
        seq.length += 1
        return blk * bs + off

    def _slots_for_append(self, seq: _Sequence, n_tokens: int) -> list:
        """Slots of the next ``n_tokens`` tokens: :meth:`_slot_for_append`, a block at a time."""
        slots = []
        while n_tokens > 0:
            first = self._slot_for_append(seq)
            more = min(n_tokens, self.block_size - first % self.block_size) - 1
            slots.extend(range(first, first + more + 1))
            seq.length += more
            n_tokens -= more + 1
        return slots

    def _upload(self, arrays: dict, wait: bool) -> dict:
        """The numpy arrays as tensors on the cache's device, in one copy from pinned memory.  Without ``wait`` the
        copy is only ordered on the current stream."""
        if self.device.type != "cuda":
            return {name: torch.from_numpy(a).to(self.device) for name, a in arrays.items()}
        starts, total = [], 0
        for a in arrays.values():
            starts.append(total)
            total += -(-a.nbytes // 16) * 16
        host = torch.empty(max(total, 16), dtype=torch.uint8, device="cpu", pin_memory=True)  # (whatever the default device)
        for start, a in zip(starts, arrays.values()):
            host.numpy()[start:start + a.nbytes] = a.reshape(-1).view(np.uint8)
        there = host.to(self.device, non_blocking=not wait)
        return {name: there[start:start + a.nbytes].view(getattr(torch, str(a.dtype))).view(a.shape)
                for start, (name, a) in zip(starts, arrays.items())}

    # ---- decoding without per-step host work ---------------------------------------------
    def reserve(self, sid: int, total_length: int) -> None:
        """Give the sequence every block it needs to grow to ``total_length``
        tokens, and un-share the block its next token goes to, so that the
        following appends need nothing from the host (a captured graph can
        compute their slots on the device from :meth:`block_table`)."""
        seq = self._seqs[sid]
        bs = self.block_size
        need = self._blocks_needed(seq, max(total_length - seq.length, 0))
        if need > self.allocator.num_free:
            raise OutOfBlocks(f"{need} KV blocks needed, {self.allocator.num_free} free")
        idx, off = divmod(seq.length, bs)
        if off and self.allocator.ref_count(seq.blocks[idx]) > 1:
            new = self.allocator.allocate()
            old = seq.blocks[idx]
            self.k_pools[:, new].copy_(self.k_pools[:, old])
            self.v_pools[:, new].copy_(self.v_pools[:, old])
            self.allocator.release(old)
            seq.blocks[idx] = new
        while len(seq.blocks) * bs < total_length:
            seq.blocks.append(self.allocator.allocate())

    def block_table(self, seq_ids: Sequence[int]) -> torch.Tensor:
        """int32 ``[n, max_blocks]`` device table of all blocks the sequences
        hold, reserved ones included (rows padded with block 0)."""
        width = max((len(self._seqs[s].blocks) for s in seq_ids), default=1) or 1
        table = [self._seqs[s].blocks + [0] * (width - len(self._seqs[s].blocks)) for s in seq_ids]
        return torch.tensor(table, dtype=torch.int32, device=self.device).view(len(seq_ids), width)

    def advance(self, seq_ids: Sequence[int], n_tokens: int) -> None:
        """Record that ``n_tokens`` rows per sequence were appended into
        reserved blocks by device-side bookkeeping."""
        for sid in seq_ids:
            seq = self._seqs[sid]
            if seq.length + n_tokens > len(seq.blocks) * self.block_size:
                raise ValueError("tokens were appended beyond the reserved blocks")
            seq.length += n_tokens

    # ---- per-step metadata -----------------------------------------------------------
    def prepare(self, seq_ids: Sequence[int], new_tokens: int | Iterable[int],
                cohort_size: int = 1) -> PagedAttentionMetadata:
        """Advance each sequence by its number of new tokens (one int for all,
        or one per sequence: the step's tensors are then ``[b, longest, ...]``
        with the rows a sequence does not have as padding, slot -1) and build
        the step's metadata.  The new K/V rows must then be passed through
        ``Attention.forward(..., kv_cache=cache.layer(l), attn_metadata=meta)``
        for every layer; the same metadata serves all layers.

        ``cohort_size`` > 1 groups consecutive ``seq_ids`` into cohorts and
        records how many leading blocks each cohort's members alias (forks of
        one prompt listed next to each other), so decode streams them once."""
        return self._prepare(seq_ids, new_tokens, cohort_size, wait=True)[0]

    def _prepare(self, seq_ids, new_tokens, cohort_size=1, wait=False):
        """:meth:`prepare` and the index int64 ``[n, longest]`` that each row of the step has in its sequence
        (padding counted on).  Without ``wait`` the tensors are for work on the current stream."""
        if self.device.type == "cuda" and torch.cuda.is_current_stream_capturing():
            # (a graph would replay this step's values)
            raise RuntimeError("the bookkeeping of a step cannot be captured: reserve() the blocks and hand the model "
                               "attn_metadata that the device keeps up to date")
        n = len(seq_ids)
        # (whole numbers of any kind: a tensor's elements, numpy's, truth values)
        counts = [int(index(c)) for c in ([new_tokens] * n if isinstance(new_tokens, int) else new_tokens)]
        if len(counts) != n:
            raise ValueError("one new-token count per sequence")
        if any(c < 0 for c in counts):
            raise ValueError("a sequence cannot have a negative number of new tokens")
        width = max(counts) if counts else 0
        ragged = any(c != width for c in counts)
        if ragged and cohort_size > 1:
            raise ValueError("cohorts are a decode feature: one new token per sequence")
        # all or nothing: a step that does not fit leaves every sequence as it was
        need = sum(self._blocks_needed(self._seqs[sid], c) for sid, c in zip(seq_ids, counts))
        if need > self.allocator.num_free:
            raise OutOfBlocks(f"{need} KV blocks needed for this step, {self.allocator.num_free} free")
        slots = np.full((n, width), -1, dtype=np.int64)
        past = np.zeros((n, 1), dtype=np.int64)
        for i, (sid, c) in enumerate(zip(seq_ids, counts)):
            seq = self._seqs[sid]
            past[i] = seq.length
            if c > 0:
                slots[i, :c] = self._slots_for_append(seq, c)
        row_index = past + np.arange(width)
        there = np.arange(width) < np.asarray(counts, dtype=np.int64).reshape(n, 1)
        lens = [self._seqs[s].length for s in seq_ids]
        max_blocks = max((len(self._seqs[s].blocks) for s in seq_ids), default=1) or 1
        table = np.zeros((n, max_blocks), dtype=np.int32)
        for row, sid in zip(table, seq_ids):
            row[:len(self._seqs[sid].blocks)] = self._seqs[sid].blocks
        arrays = {"slots": slots.reshape(-1), "index": row_index, "table": table, "lens": np.asarray(lens, dtype=np.int32),
                  "positions": np.where(there, row_index, 0).astype(np.int32).reshape(-1)}
        if ragged:
            # rows are padded to `width` ([b, width, ...] tensors); the kernels get the true bounds
            # and the layer packs the rows that exist
            arrays["cu"] = np.cumsum([0] + counts).astype(np.int32)
            arrays["rows"] = np.flatnonzero(there).astype(np.int64)
        if cohort_size > 1 and n > 0:
            from .paged_ops import shared_prefix_blocks
            arrays["shared"] = np.ascontiguousarray(
                shared_prefix_blocks(table.tolist(), lens, self.block_size, cohort_size))
        t = self._upload(arrays, wait)
        return PagedAttentionMetadata(
            block_tables=t["table"], context_lens=t["lens"], slot_mapping=t["slots"],
            max_context_len=max(lens, default=0), cu_seqlens_q=t.get("cu"),
            cohort_size=cohort_size if "shared" in t else 1, cohort_shared_blocks=t.get("shared"),
            positions=t["positions"], chunk_rows=t.get("rows"), max_chunk_len=width), t["index"]
