"""The prefill kernel for long sweeps (256-row workgroups, 16 bits, head dim
128) against the oracle in the element type and in float64: both types, grouped
queries, last query tiles and K/V tiles that are partly filled, block sizes that
are no power of two, more sequences than are ranked, unused pool slots that hold
NaN, no causal rule, dense calls without tables.  Each case asserts by name that
this kernel ran: the line between the two prefill kernels may move, the cases
have to move with it.  (The line looks at the width of the block table, so wide
tables bring short contexts here.)"""
import pytest
import torch

from ironcore_amd import config as ic_config, paged_ops, workloads
from ironcore_amd.layers import Attention
from oracle import paged as oracle_paged
from oracle.dense_attention import causal_offset_mask, dense_attention
from parity_bars import hold

pytestmark = pytest.mark.gpu


def _on_the_long_kernel(call):
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA], acc_events=True) as prof:
        out = call()
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    assert "paged_prefill_kernel" in names and "paged_prefill_short_kernel" not in names, names
    return out


def _hold(wl, gpu, causal=True):
    width = -(-2304 // wl.block_size)
    tables = torch.zeros(len(wl.chunk_lens), max(width, wl.block_tables.shape[1]), dtype=torch.int32)
    tables[:, :wl.block_tables.shape[1]] = wl.block_tables
    d = wl.to(gpu)
    paged_ops.kv_append(d.k_new, d.v_new, d.k_pool, d.v_pool, d.slot_mapping)
    out = _on_the_long_kernel(lambda: paged_ops.paged_prefill(
        d.query, d.k_pool, d.v_pool, tables.to(gpu), d.context_lens, d.cu_seqlens_q, d.max_chunk_len, causal=causal))
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,hn,gn,prefix,chunks", [
    (9, 16, 16, (0, 70), (225, 256)), (9, 16, 4, (0, 70), (225, 256)), (10, 14, 2, (30, 90), (250, 256)),
    (5, 16, 16, (0, 50), (481, 512)), (5, 16, 2, (0, 300), (481, 512)),    # two query tiles, the second partly filled
    (9, 16, 16, (0, 0), (1, 256)), (70, 2, 1, (0, 40), (1, 256))])         # ragged; more sequences than are ranked
def test_chunks(gpu, dtype, n, hn, gn, prefix, chunks):
    wl = workloads.make_prefill_workload(n, hn, gn, 128, *prefix, *chunks, dtype=dtype, seed=hn + gn + chunks[0])
    _hold(wl, gpu)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block", [48, 64, 112])
def test_block_sizes(gpu, dtype, block):
    wl = workloads.make_prefill_workload(9, 16, 4, 128, 0, 100, 225, 256, block_size=block, dtype=dtype, seed=block)
    _hold(wl, gpu)


@pytest.mark.parametrize("hn,gn", [(16, 16), (16, 4)])
def test_long_prefixes(gpu, hn, gn):
    wl = workloads.make_prefill_workload(9, hn, gn, 128, 1000, 1400, 240, 256, seed=hn + gn)
    _hold(wl, gpu)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_nan_in_unused_slots(gpu, dtype):
    wl = workloads.make_prefill_workload(9, 16, 4, 128, 0, 100, 225, 256, dtype=dtype, seed=5)
    for table, ctx in zip(wl.block_tables, wl.context_lens.tolist()):
        if ctx % 16:
            last = int(table[(ctx - 1) // 16])
            wl.k_pool[last, :, ctx % 16:] = float("nan")
            wl.v_pool[last, :, ctx % 16:] = float("nan")
    _hold(wl, gpu)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hn,gn", [(16, 16), (16, 4)])
def test_no_causal_rule(gpu, dtype, hn, gn):
    wl = workloads.make_prefill_workload(9, hn, gn, 128, 0, 100, 225, 256, dtype=dtype, seed=hn + gn)
    _hold(wl, gpu, causal=False)


@pytest.mark.parametrize("dtype,precision,b,sq,sk,hn,gn,causal", [
    (torch.bfloat16, "bf16", 1, 2048, 2048, 16, 16, True), (torch.bfloat16, "bf16", 1, 2048, 2048, 16, 16, False),
    (torch.bfloat16, "bf16", 5, 512, 2201, 16, 4, False), (torch.float16, "fp16", 5, 500, 1301, 16, 16, True)])
def test_dense_calls(gpu, dtype, precision, b, sq, sk, hn, gn, causal):
    g = torch.Generator().manual_seed(sk)
    q, k, v = (torch.randn(b, n, h, 128, generator=g).to(dtype) for n, h in ((sq, hn), (sk, gn), (sk, gn)))
    mask = causal_offset_mask(sq, sk) if causal else None
    attn = Attention(ic_config.MainConfig(
        model=ic_config.ModelConfig(d_model=hn * 128, num_attention_heads=hn, num_attention_groups=gn, head_dim=128,
                                    dropout_attn=0.0, precision=precision),
        trainer=ic_config.TrainerConfig(use_flash_attn=False))).eval()
    given = tuple(t.to(gpu) for t in (q, k, v)) + (None if mask is None else mask.to(gpu),)
    out = _on_the_long_kernel(lambda: attn(*given))
    fewest = sk - sq + 1 if causal else sk
    hold(out, dense_attention(q, k, v, mask), dense_attention(q.double(), k.double(), v.double(), mask), dtype, fewest)
