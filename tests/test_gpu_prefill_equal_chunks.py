"""Chunks of one length need no bounds array: the layer call without one against the call with it, bit for bit, for one
sequence to more than the kernels rank at once, all types (each has its kernel), and what the descriptor still refuses."""
import ctypes

import numpy as np
import pytest
import torch

from ironcore_amd import _lib
from ironcore_amd import config as ic_config
from ironcore_amd.layers import Attention, PagedAttentionMetadata, RotaryPositionalEmbedding

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,chunk,prefix,rope", [(1, 2, 0, False), (3, 33, 50, True), (65, 20, 30, False), (2, 600, 700, False)])
def test_without_bounds(gpu, dtype, n, chunk, prefix, rope):
    hn, gn, hd, block = 4, 2, 64, 16
    cfg = ic_config.MainConfig(model=ic_config.ModelConfig(d_model=hn * hd, num_attention_heads=hn, num_attention_groups=gn,
                                                           head_dim=hd, dropout_attn=0.0),
                               trainer=ic_config.TrainerConfig(use_flash_attn=False))
    layer = Attention(cfg).to(gpu).eval()
    g = torch.Generator().manual_seed(n)
    past = [prefix * i // n for i in range(n)]
    blocks = [-(-(p + chunk) // block) for p in past]
    tables = np.zeros((n, max(blocks)), dtype=np.int32)
    perm, at = torch.randperm(sum(blocks), generator=g).numpy(), 0
    slots, positions = [], []
    for i, p in enumerate(past):
        tables[i, :blocks[i]] = perm[at:at + blocks[i]]
        at += blocks[i]
        pos = np.arange(p, p + chunk)
        positions.append(pos)
        slots.append(tables[i, pos // block].astype(np.int64) * block + pos % block)
    q, k, v = (torch.randn(n, chunk, h, hd, generator=g).to(dtype).to(gpu) for h in (hn, gn, gn))
    pools = [torch.randn(sum(blocks), gn, block, hd, generator=g).to(dtype).to(gpu) for _ in range(2)]
    out = []
    for cu in (None, torch.arange(0, (n + 1) * chunk, chunk, dtype=torch.int32, device=gpu)):
        meta = PagedAttentionMetadata(
            block_tables=torch.from_numpy(tables).to(gpu),
            context_lens=torch.tensor([p + chunk for p in past], dtype=torch.int32, device=gpu),
            slot_mapping=torch.from_numpy(np.concatenate(slots)).to(gpu), max_context_len=max(past) + chunk, cu_seqlens_q=cu,
            positions=torch.from_numpy(np.concatenate(positions).astype(np.int32)).to(gpu))
        mine = [t.clone() for t in pools]
        with torch.no_grad():
            out.append([layer(q, k, v, None, kv_cache=tuple(mine), attn_metadata=meta,
                              rotary_pos_emb=RotaryPositionalEmbedding(hd, max_seq_len=2000).to(gpu) if rope else None), *mine])
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_what_the_descriptor_refuses(gpu):
    lib = _lib.load()
    t = torch.zeros(4, 1, 16, 64, device=gpu)
    ints = torch.zeros(4, dtype=torch.int32, device=gpu)

    def call(**over):
        c = dict(out=t.data_ptr(), out_stride_token=64, q=t.data_ptr(), q_stride_token=64, k_pool=t.data_ptr(), v_pool=t.data_ptr(),
                 pool_stride_block=1024, pool_stride_head=1024, pool_stride_token=64, block_tables=ints.data_ptr(),
                 block_table_stride=2, context_lens=ints.data_ptr(), n_seqs=2, max_chunk_len=8, hn=1, gn=1, hd=64, block_size=16,
                 num_blocks=4, scale=1.0, causal=1, dtype=2)
        return lib.ic_paged_prefill_ex(ctypes.byref(_lib.STRUCTS["ic_prefill_call"](**{**c, **over})), 0)
    assert call() < 0                                                    # neither bounds nor a pitch
    assert call(row_pitch=7) < 0                                         # chunks that overlap
    assert call(row_pitch=8, cu_seqlens_q=ints.data_ptr()) < 0           # both
    assert call(row_pitch=8, rows=t.data_ptr(), n_rows=4, q_rows=16) < 0
