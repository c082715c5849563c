"""Small batches of short contexts (paged_decode_pair_kernel): contexts at the
edges of tiles and rounds, group sizes that fill a wave's heads or not, blocks
of several tiles, an empty sequence, unused pool rows that hold NaN; against the
oracle and against the split path (reached through min_chunk_tokens)."""
import pytest
import torch

from ironcore_amd import paged_ops, workloads
from oracle import paged as oracle_paged

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2e-2, torch.float16: 3e-3, torch.float32: 1e-5}


def _run(wl, gpu, **kw):
    d = wl.to(gpu)
    return paged_ops.paged_decode(d.query, d.k_pool, d.v_pool, d.block_tables, d.context_lens, d.max_context_len,
                                  **kw).cpu()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hn,gn,hd,block", [(12, 12, 64, 16), (4, 2, 128, 48), (6, 2, 128, 16), (8, 2, 32, 16),
                                            (4, 4, 32, 32)])
def test_edges(gpu, dtype, hn, gn, hd, block):
    lens = (1, 15, 16, 17, 128, 129, 0, 255)
    wl = workloads.make_decode_workload(len(lens), hn, gn, hd, 255, 255, block_size=block, dtype=dtype, seed=hn + hd)
    wl.context_lens = torch.tensor(lens, dtype=torch.int32)
    alive = [i for i, n in enumerate(lens) if n]
    ref = oracle_paged.paged_decode(wl.query[alive], wl.k_pool, wl.v_pool, wl.block_tables[alive],
                                    wl.context_lens[alive])
    for i, n in enumerate(lens):                                # rows past a context may hold anything
        for j in range(n, wl.block_tables.shape[1] * block):
            wl.k_pool[wl.block_tables[i, j // block], :, j % block] = float("nan")
            wl.v_pool[wl.block_tables[i, j // block], :, j % block] = float("nan")
    out = _run(wl, gpu)
    assert not out[lens.index(0)].any()
    assert (out[alive].float() - ref.float()).abs().max().item() <= TOL[dtype]
    split = _run(wl, gpu, min_chunk_tokens=32)
    # one rounding apart (16 bits: 2^-8 of values up to 4, where a context is one token)
    assert torch.allclose(out.float(), split.float(), rtol=TOL[dtype], atol=4e-3 if dtype != torch.float32 else 1e-5)


def test_table_entries_out_of_the_pool_are_clamped(gpu):
    wl = workloads.make_decode_workload(2, 4, 4, 64, 100, 100, dtype=torch.float32, seed=4)
    want = wl.block_tables.clone()
    want[0, 1], want[1, 2] = 0, wl.k_pool.shape[0] - 1
    wl.block_tables[0, 1], wl.block_tables[1, 2] = -7, 10 ** 6
    ref = oracle_paged.paged_decode(wl.query, wl.k_pool, wl.v_pool, want, wl.context_lens)
    assert (_run(wl, gpu) - ref).abs().max().item() <= TOL[torch.float32]


@pytest.mark.parametrize("dtype,hn,gn,hd", [(torch.bfloat16, 4, 4, 128), (torch.bfloat16, 6, 6, 64), (torch.float32, 3, 3, 64),
                                            (torch.float16, 4, 2, 64), (torch.bfloat16, 4, 2, 128), (torch.bfloat16, 8, 2, 64)])
@pytest.mark.parametrize("longest", [1024, 1025, 1280, 1281, 2047, 2048, 2049])
def test_rounds_up_to_the_limits(gpu, dtype, hn, gn, hd, longest):
    """Contexts of 8 to 16 rounds, and past what the pair kernel takes (fewer rounds with wide rows or grouped heads)."""
    lens = (longest, 1, longest - 127, longest // 2, 129)
    wl = workloads.make_decode_workload(len(lens), hn, gn, hd, longest, longest, dtype=dtype, seed=longest)
    wl.context_lens = torch.tensor(lens, dtype=torch.int32)
    ref = oracle_paged.paged_decode(wl.query, wl.k_pool, wl.v_pool, wl.block_tables, wl.context_lens)
    assert (_run(wl, gpu).float() - ref.float()).abs().max().item() <= TOL[dtype]


@pytest.mark.parametrize("batch,hn,gn,hd,dtype", [
    (300, 4, 4, 64, torch.bfloat16), (700, 4, 2, 64, torch.float16), (300, 3, 3, 64, torch.float32),
    (127, 16, 4, 64, torch.bfloat16), (129, 16, 4, 64, torch.bfloat16)])      # 508 and 516 pairs: the pair kernel's, the split's
def test_large_batches(gpu, batch, hn, gn, hd, dtype):
    wl = workloads.make_decode_workload(batch, hn, gn, hd, 1, 300, dtype=dtype, seed=batch)
    ref = oracle_paged.paged_decode(wl.query, wl.k_pool, wl.v_pool, wl.block_tables, wl.context_lens)
    assert (_run(wl, gpu).float() - ref.float()).abs().max().item() <= TOL[dtype]
