"""The prefill kernel for short work (32-row wave blocks of several heads in a
workgroup; two tile groups where the grid leaves a CU one workgroup) at the
edges of its blocks, tiles and launch rules, against the oracle in the element
type and in float64."""
import pytest
import torch

from ironcore_amd import paged_ops, workloads
from oracle import paged as oracle_paged
from oracle.dense_attention import dense_attention
from parity_bars import hold

pytestmark = pytest.mark.gpu


def _hold(wl, gpu, causal=True):
    d = wl.to(gpu)
    paged_ops.kv_append(d.k_new, d.v_new, d.k_pool, d.v_pool, d.slot_mapping)
    out = paged_ops.paged_prefill(d.query, d.k_pool, d.v_pool, d.block_tables, d.context_lens, d.cu_seqlens_q,
                                  d.max_chunk_len, causal=causal)
    torch.cuda.synchronize()
    kp, vp = d.k_pool.cpu(), d.v_pool.cpu()

    def oracle(dtype):
        q, k, v = wl.query.to(dtype), kp.to(dtype), vp.to(dtype)
        if causal:
            return oracle_paged.paged_prefill(q, k, v, wl.block_tables, wl.context_lens, wl.cu_seqlens_q)
        return torch.cat([dense_attention(
            q[wl.cu_seqlens_q[i]:wl.cu_seqlens_q[i + 1]][None],
            oracle_paged.gather_kv(k, wl.block_tables[i], int(n)), oracle_paged.gather_kv(v, wl.block_tables[i], int(n)),
            None)[0] for i, n in enumerate(wl.context_lens)])

    fewest = int(wl.context_lens.min()) if not causal else min(wl.prefix_lens) + 1
    hold(out, oracle(wl.query.dtype), oracle(torch.float64), wl.query.dtype, fewest)


@pytest.mark.parametrize("chunk", [1, 31, 32, 33, 64, 127, 129, 257])
@pytest.mark.parametrize("hn,gn,hd", [(2, 2, 128), (6, 2, 64), (7, 1, 128), (8, 1, 32)])
def test_chunk_edges(gpu, chunk, hn, gn, hd):
    wl = workloads.make_prefill_workload(2, hn, gn, hd, 0, 100, chunk, chunk, seed=chunk + hd)
    _hold(wl, gpu)


@pytest.mark.parametrize("prefix", [0, 448, 513, 1100])       # either side of the line from which tile groups are used
@pytest.mark.parametrize("chunk", [5, 63, 65, 128])
@pytest.mark.parametrize("hd,dtype", [(128, torch.bfloat16), (64, torch.float16)])
def test_two_tile_groups(gpu, prefix, chunk, hd, dtype):
    wl = workloads.make_prefill_workload(1, 4, 2, hd, prefix, prefix, chunk, chunk, dtype=dtype, seed=prefix + chunk)
    _hold(wl, gpu)


@pytest.mark.parametrize("n_seqs,hn,gn,hd,block", [(22, 12, 12, 32, 16),    # 264 workgroups: the slices of the second half
                                                   (9, 32, 8, 64, 48),     # flip their blocks' order
                                                   (70, 8, 1, 128, 16)])   # more sequences than are ranked
def test_grids_beyond_one_workgroup_per_cu(gpu, n_seqs, hn, gn, hd, block):
    wl = workloads.make_prefill_workload(n_seqs, hn, gn, hd, 0, 40, 1, 140, block_size=block, seed=n_seqs)
    _hold(wl, gpu)


@pytest.mark.parametrize("chunk,prefix", [(40, 0), (40, 600)])
def test_no_causal_rule_and_empty_chunks(gpu, chunk, prefix):
    wl = workloads.make_prefill_workload(3, 6, 2, 128, prefix, prefix, chunk, chunk, seed=chunk)
    _hold(wl, gpu, causal=False)
    wl = workloads.make_prefill_workload(5, 6, 2, 128, prefix, prefix, 0, 3, seed=chunk + 1)
    _hold(wl, gpu)


@pytest.mark.parametrize("hn,gn,hd,n_seqs,chunk,prefix,causal", [
    (4, 4, 128, 2, 64, 0, True), (2, 2, 128, 1, 300, 16, True), (2, 2, 128, 1, 300, 32, True),      # 64, 320 tokens
    (4, 4, 128, 2, 33, 80, False), (4, 4, 128, 2, 33, 96, False),                                   # 128
    (12, 12, 64, 85, 70, 0, True), (12, 12, 64, 86, 70, 0, True), (4, 4, 64, 64, 70, 0, False), (4, 4, 64, 65, 70, 0, False),
    # grouped: 512 tokens, a workgroup to a CU; a workgroup of two heads' and of three heads' blocks
    (8, 2, 64, 2, 100, 412, True), (8, 2, 64, 2, 100, 413, True), (8, 2, 64, 2, 33, 0, True), (6, 2, 64, 3, 70, 9, False),
    (8, 2, 128, 2, 4, 700, True), (8, 2, 128, 2, 5, 700, True), (4, 4, 128, 2, 8, 700, False), (4, 4, 128, 2, 9, 700, False),
    (8, 1, 32, 1, 20, 0, True), (8, 2, 128, 2, 100, 0, True), (8, 2, 128, 2, 120, 9, True), (16, 2, 64, 40, 70, 0, True)])
def test_rows_moved_directly_and_whole(gpu, hn, gn, hd, n_seqs, chunk, prefix, causal):
    """Either side of the lines between the two ways in which query rows and outputs move."""
    wl = workloads.make_prefill_workload(n_seqs, hn, gn, hd, prefix, prefix, chunk, chunk, seed=n_seqs + chunk)
    _hold(wl, gpu, causal=causal)
