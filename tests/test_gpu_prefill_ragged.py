"""Chunks of unequal length (rows named one by one): workgroups numbered over all sequences by the length of their
sweep, against the same chunks numbered sequence by sequence; the append's launch with the zeroing beside it."""
import ctypes
import json

import pytest
import torch

from ironcore_amd import _lib, paged_ops, workloads
from ironcore_amd.layers import RotaryPositionalEmbedding

pytestmark = pytest.mark.gpu

Prefill = _lib.STRUCTS["ic_prefill_call"]
Append = _lib.STRUCTS["ic_append_call"]


def _attend(d, hn, gn, hd, causal, rows, positions, emb, out, q):
    call = Prefill(out=out.data_ptr(), out_stride_token=hn * hd, q=q.data_ptr(), q_stride_token=hn * hd,
                   k_pool=d.k_pool.data_ptr(), v_pool=d.v_pool.data_ptr(), pool_stride_block=d.k_pool.stride(0),
                   pool_stride_head=d.k_pool.stride(1), pool_stride_token=d.k_pool.stride(2), block_tables=d.block_tables.data_ptr(),
                   block_table_stride=d.block_tables.stride(0), context_lens=d.context_lens.data_ptr(),
                   cu_seqlens_q=d.cu_seqlens_q.data_ptr(), n_seqs=len(d.context_lens), max_chunk_len=d.max_chunk_len, hn=hn, gn=gn,
                   hd=hd, block_size=d.k_pool.shape[2], num_blocks=d.k_pool.shape[0], scale=hd ** -0.5, causal=causal,
                   dtype=_lib.IC_DTYPE[q.dtype])
    if rows is not None:
        call.rows, call.n_rows, call.q_rows = rows.data_ptr(), rows.numel(), q.shape[0]
    if emb is not None:
        call.positions, call.cos_table, call.sin_table = positions.data_ptr(), emb.cos_emb.data_ptr(), emb.sin_emb.data_ptr()
        call.table_rows = emb.cos_emb.shape[0]
    assert _lib.load().ic_paged_prefill_ex(ctypes.byref(call), _lib.current_stream_ptr(q.device)) == 0
    return out


@pytest.mark.parametrize("n_seqs,hn,gn,hd,block,prefix,chunks,dtype", [
    (1, 7, 1, 128, 16, (0, 0), (97, 97), torch.bfloat16),      # one sequence, a group that fills no workgroup
    (16, 8, 8, 128, 16, (0, 200), (0, 300), torch.bfloat16),   # as many as a row of lanes holds; empty chunks
    (17, 4, 2, 64, 48, (0, 700), (1, 65), torch.float16),
    (64, 6, 2, 32, 16, (0, 40), (0, 140), torch.bfloat16),     # a sequence to every lane
    (65, 6, 2, 64, 16, (0, 40), (1, 70), torch.bfloat16),      # one more: numbered sequence by sequence
    (3, 28, 4, 128, 16, (1500, 1600), (1, 130), torch.bfloat16),
    (9, 12, 12, 128, 16, (0, 0), (3, 700), torch.bfloat16),
    # more workgroups to an XCD than it holds: 36, 40 and up to 44 of one unit; 16 units of 5 and of 9
    (1, 36, 1, 128, 16, (0, 0), (97, 97), torch.bfloat16),
    (3, 64, 4, 128, 16, (1500, 1600), (290, 500), torch.bfloat16),
    (17, 48, 2, 64, 48, (0, 700), (1, 220), torch.float16),
    (16, 8, 8, 128, 16, (0, 200), (0, 600), torch.bfloat16),
    (64, 6, 2, 32, 16, (0, 40), (0, 340), torch.bfloat16)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("rope", [False, True])
def test_by_sweep(gpu, n_seqs, hn, gn, hd, block, prefix, chunks, dtype, causal, rope):
    wl = workloads.make_prefill_workload(n_seqs, hn, gn, hd, *prefix, *chunks, block_size=block, dtype=dtype, seed=n_seqs)
    d = wl.to(gpu)
    paged_ops.kv_append(d.k_new, d.v_new, d.k_pool, d.v_pool, d.slot_mapping)
    if not causal and n_seqs > 1:
        d.context_lens[n_seqs // 2] = 0        # rows without a key: zeros
    total = d.query.shape[0]
    emb = RotaryPositionalEmbedding(hd, max_seq_len=300).to(gpu) if rope else None
    g = torch.Generator().manual_seed(n_seqs)
    positions = torch.randint(-2, 320, (total,), generator=g, dtype=torch.int32).to(gpu)
    want = torch.empty(total, hn * hd, dtype=dtype, device=gpu)
    _attend(d, hn, gn, hd, causal, None, positions, emb, want, d.query)
    spread = torch.randperm(2 * total + 3, generator=g)[:total].to(gpu)                   # any rows of a larger tensor
    q = torch.full((2 * total + 3, hn, hd), float("nan"), dtype=dtype, device=gpu)
    q[spread] = d.query
    at = torch.full((2 * total + 3,), -1, dtype=torch.int32, device=gpu)
    at[spread] = positions
    out = torch.full((2 * total + 3, hn * hd), 7.0, dtype=dtype, device=gpu)
    _attend(d, hn, gn, hd, causal, spread, at, emb, out, q)
    # the same sums, in two tile groups or one: a rounding of the result apart
    assert torch.allclose(out[spread].float(), want.float(), rtol=2 ** -7, atol=2 ** -9)
    untouched = torch.ones(2 * total + 3, dtype=torch.bool, device=gpu)
    untouched[spread] = False
    assert (out[untouched] == 7).all()


@pytest.mark.parametrize("hn,gn,hd,dtype", [(4, 4, 128, torch.bfloat16), (14, 2, 128, torch.float16), (6, 2, 64, torch.bfloat16),
                                            (4, 4, 32, torch.float16)])
@pytest.mark.parametrize("rows", [1, 4, 5, 8, 9])
@pytest.mark.parametrize("named", [False, True])
def test_few_rows_rotated_on_their_way(gpu, hn, gn, hd, dtype, rows, named):
    """Either side of the lines from which rotated query rows move as whole rows: the same bits as rows rotated before."""
    wl = workloads.make_prefill_workload(3, hn, gn, hd, 0, 90, rows if not named else 1, rows, dtype=dtype, seed=rows)
    wl.max_chunk_len = rows
    d = wl.to(gpu)
    paged_ops.kv_append(d.k_new, d.v_new, d.k_pool, d.v_pool, d.slot_mapping)
    total = d.query.shape[0]
    emb = RotaryPositionalEmbedding(hd, max_seq_len=100).to(gpu)
    positions = torch.arange(total, dtype=torch.int32, device=gpu) * 7 - 2                       # clamped into the table
    list_of_rows = torch.arange(total, device=gpu) if named else None
    got, want = (torch.empty(total, hn * hd, dtype=dtype, device=gpu) for _ in range(2))
    _attend(d, hn, gn, hd, True, list_of_rows, positions, emb, got, d.query)
    before = emb(d.query.view(1, total, hn, hd), positions.clamp(min=0)).view(total, hn, hd)
    _attend(d, hn, gn, hd, True, list_of_rows, positions, None, want, before)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n_seqs,width,gn,hd", [(1, 5, 1, 32), (3, 40, 2, 64), (2, 70, 33, 128)])
@pytest.mark.parametrize("rope", [False, True])
def test_append_and_zeroing(gpu, dtype, n_seqs, width, gn, hd, rope):
    g = torch.Generator(device=gpu).manual_seed(width)
    n = n_seqs * width
    k, v = (torch.randn(n, gn, hd, generator=g, device=gpu).to(dtype) for _ in range(2))
    lens = [width - 3 * i for i in range(n_seqs)]
    rows = torch.tensor([i * width + t for i, c in enumerate(lens) for t in range(c)], device=gpu)
    bounds = torch.tensor([0] + lens, dtype=torch.int32, device=gpu).cumsum(0, dtype=torch.int32)
    slots = torch.full((n,), -1, dtype=torch.int64, device=gpu)
    slots[rows] = torch.randperm(160, device=gpu, generator=g)[:len(rows)]
    positions = torch.randint(0, 90, (n,), generator=g, device=gpu, dtype=torch.int32)
    emb = RotaryPositionalEmbedding(hd, max_seq_len=90).to(gpu)
    pools = [torch.zeros(10, gn, 16, hd, dtype=dtype, device=gpu) for _ in range(4)]
    if rope:
        paged_ops.rope_kv_append(torch.zeros(n, 1, hd, dtype=dtype, device=gpu), k, v, pools[0], pools[1], slots, positions,
                                 emb.cos_emb, emb.sin_emb)
    else:
        paged_ops.kv_append(k, v, pools[0], pools[1], slots)
    out = torch.full((n, 3 * hd), 7.0, dtype=dtype, device=gpu)
    call = Append(k_new=k.data_ptr(), v_new=v.data_ptr(), new_stride_token=gn * hd, k_pool=pools[2].data_ptr(),
                  v_pool=pools[3].data_ptr(), pool_stride_block=gn * 16 * hd, pool_stride_head=16 * hd, pool_stride_token=hd,
                  num_blocks=10, slot_mapping=slots.data_ptr(), n_tokens=n, gn=gn, hd=hd, block_size=16,
                  dtype=_lib.IC_DTYPE[dtype], positions=positions.data_ptr(), table_rows=90, zero_out=out.data_ptr(),
                  zero_stride_bytes=3 * hd * k.element_size(), rows=rows.data_ptr(), n_rows=len(rows), bounds=bounds.data_ptr(),
                  zero_row_bytes=3 * hd * k.element_size(), n_seqs=n_seqs, row_pitch=width)
    if rope:
        call.cos_table, call.sin_table = emb.cos_emb.data_ptr(), emb.sin_emb.data_ptr()
    assert _lib.load().ic_append_chunks(ctypes.byref(call), _lib.current_stream_ptr(gpu)) == 0
    assert torch.equal(pools[0], pools[2]) and torch.equal(pools[1], pools[3])
    listed = torch.zeros(n, dtype=torch.bool, device=gpu)
    listed[rows] = True
    assert (out[listed] == 7).all() and not out[~listed].any()


def _padded(gpu, n_seqs, width, lens):
    """(a padded output to zero, the rows that exist, their bounds, which rows those are)"""
    rows = torch.tensor([i * width + t for i, c in enumerate(lens) for t in range(c)], dtype=torch.int64, device=gpu)
    bounds = torch.tensor([0] + list(lens), dtype=torch.int32, device=gpu).cumsum(0, dtype=torch.int32)
    listed = torch.zeros(n_seqs * width, dtype=torch.bool, device=gpu)
    listed[rows] = True
    return torch.full((n_seqs * width, 72), 7.0, dtype=torch.bfloat16, device=gpu), rows, bounds, listed


@pytest.mark.parametrize("width,lens", [(1, (0, 1, 0)), (5, (5, 0, 2)), (40, (0, 0, 0)), (1200, (1200, 3, 700))])
def test_zeroing_alone(gpu, width, lens):
    """The entry point without an append; rows wider than what is zeroed keep the rest."""
    out, rows, bounds, listed = _padded(gpu, len(lens), width, lens)
    rows = torch.cat([rows, rows.new_full((1,), -5)])         # (an address for the list without entries)
    assert _lib.load().ic_zero_unlisted_rows(out.data_ptr(), 144, 128, rows.data_ptr(), len(rows) - 1, bounds.data_ptr(),
                                             len(lens), width, _lib.current_stream_ptr(gpu)) == 0
    assert (out[listed] == 7).all() and not out[~listed][:, :64].any() and (out[:, 64:] == 7).all()


@pytest.mark.parametrize("tokens", [0, 6])
@pytest.mark.parametrize("lens", [(2, 1), (0, 0)])
def test_zeroing_without_tokens_or_listed_rows(gpu, tokens, lens):
    """The zeroing is done whether or not there is a token to append or a row that a chunk holds."""
    out, rows, bounds, listed = _padded(gpu, 2, 3, lens)
    k = torch.randn(6, 2, 32, device=gpu).bfloat16()
    pool = torch.zeros(1, 2, 16, 32, dtype=torch.bfloat16, device=gpu)
    slots = torch.arange(6, device=gpu)
    call = Append(k_new=k.data_ptr(), v_new=k.data_ptr(), new_stride_token=64, k_pool=pool.data_ptr(), v_pool=pool.data_ptr(),
                  pool_stride_block=1024, pool_stride_head=512, pool_stride_token=32, num_blocks=1,
                  slot_mapping=slots.data_ptr(), n_tokens=tokens, gn=2, hd=32, block_size=16, dtype=0,
                  zero_out=out.data_ptr(), zero_stride_bytes=144, rows=rows.data_ptr() if len(rows) else None,
                  n_rows=len(rows), bounds=bounds.data_ptr(), zero_row_bytes=144, n_seqs=2, row_pitch=3)
    lib, stream = _lib.load(), _lib.current_stream_ptr(gpu)
    assert lib.ic_append_chunks(ctypes.byref(call), stream) == 0
    assert (out[listed] == 7).all() and not out[~listed].any()
    assert torch.equal(pool[0, :, :tokens], k[:tokens].transpose(0, 1)) and not pool[0, :, tokens:].any()
    call.rows, call.n_rows = None, 3                           # rows that are counted but not given
    assert lib.ic_append_chunks(ctypes.byref(call), stream) == -1


@pytest.mark.parametrize("gn,hd", [(1, 64), (1, 32), (8, 128)])
def test_zeroing_has_workgroups_of_its_own(gpu, tmp_path, gn, hd):
    """Beside an append of any width the padding rows get a workgroup each: not the few that a narrow append has."""
    from torch.profiler import ProfilerActivity, profile
    n, rows = 120, 2 * 60
    out, listed, bounds, _ = _padded(gpu, 2, 60, (60, 3))
    k = torch.randn(n, gn, hd, device=gpu).bfloat16()
    pool = torch.zeros(8, gn, 16, hd, dtype=torch.bfloat16, device=gpu)
    slots = torch.arange(n, device=gpu)
    call = Append(k_new=k.data_ptr(), v_new=k.data_ptr(), new_stride_token=gn * hd, k_pool=pool.data_ptr(), v_pool=pool.data_ptr(),
                  pool_stride_block=gn * 16 * hd, pool_stride_head=16 * hd, pool_stride_token=hd, num_blocks=8,
                  slot_mapping=slots.data_ptr(), n_tokens=n, gn=gn, hd=hd, block_size=16, dtype=0, zero_out=out.data_ptr(),
                  zero_stride_bytes=144, rows=listed.data_ptr(), n_rows=63, bounds=bounds.data_ptr(), zero_row_bytes=144,
                  n_seqs=2, row_pitch=60)
    with profile(activities=[ProfilerActivity.CUDA], acc_events=True) as prof:
        assert _lib.load().ic_append_chunks(ctypes.byref(call), _lib.current_stream_ptr(gpu)) == 0
        torch.cuda.synchronize()
    prof.export_chrome_trace(str(tmp_path / "trace.json"))
    grids = [e["args"]["grid"] for e in json.loads((tmp_path / "trace.json").read_text())["traceEvents"]
             if e.get("cat") == "kernel" and "kv_append_kernel" in e["name"]]
    assert len(grids) == 1 and grids[0][0] * grids[0][1] * (grids[0][2] - 2) >= rows, grids
