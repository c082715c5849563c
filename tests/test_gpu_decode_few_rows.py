"""Decode batches of few rows, whose pairs are cut over many waves: the reduce
pass that merges a pair's partials in slices, at both sides of the line from
which it is used, against the oracle and against one share per pair."""
import pytest
import torch

from ironcore_amd import paged_ops, workloads
from oracle import paged as oracle_paged

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2e-2, torch.float16: 2e-2, torch.float32: 1e-4}


def _run(wl, gpu, **kw):
    d = wl.to(gpu)
    out = paged_ops.paged_decode(d.query, d.k_pool, d.v_pool, d.block_tables, d.context_lens, d.max_context_len, **kw)
    torch.cuda.synchronize()
    return out.cpu()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hn,gn,hd", [(8, 8, 128), (32, 4, 128), (24, 2, 64), (7, 1, 32)])
@pytest.mark.parametrize("batch,lo,hi", [(1, 193, 193), (1, 3000, 3000), (3, 1, 2500)])
def test_few_rows_many_partials(gpu, dtype, hn, gn, hd, batch, lo, hi):
    wl = workloads.make_decode_workload(batch, hn, gn, hd, lo, hi, dtype=dtype, seed=hn + hd + batch)
    out = _run(wl, gpu)
    ref = oracle_paged.paged_decode(wl.query, wl.k_pool, wl.v_pool, wl.block_tables, wl.context_lens)
    assert torch.isfinite(out.float()).all()
    assert (out.float() - ref.float()).abs().max().item() <= TOL[dtype]
    one = _run(wl, gpu, min_chunk_tokens=1 << 20)   # one wave walks everything: no partials to merge
    assert (out.float() - one.float()).abs().max().item() <= (4e-3 if dtype != torch.float32 else 1e-5)


def test_few_rows_with_an_empty_sequence_and_cohorts(gpu):
    """A cohort of two samples behind a long prompt (two sources of partials per
    row), and an empty sequence beside a long one."""
    wl = workloads.make_grpo_workload(1, 2, 8, 2, 128, 1600, 1, 900, seed=3)
    plain = _run(wl, gpu)
    shared = torch.from_numpy(paged_ops.shared_prefix_blocks(wl.block_tables, wl.context_lens, 16, 2)).to(gpu)
    both = _run(wl, gpu, cohort_size=2, cohort_shared_blocks=shared)
    ref = oracle_paged.paged_decode(wl.query, wl.k_pool, wl.v_pool, wl.block_tables, wl.context_lens)
    assert (both.float() - ref.float()).abs().max().item() <= 2e-2
    assert (both.float() - plain.float()).abs().max().item() <= 4e-3
    wl.context_lens[0] = 0
    out = _run(wl, gpu)
    assert (out[0] == 0).all() and (out[1].float() - ref[1].float()).abs().max().item() <= 2e-2
