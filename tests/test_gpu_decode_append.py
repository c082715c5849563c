"""A decode step's append inside the attention launch (paged_decode_pair_kernel, APPEND): the same bits, in
outputs and pools, as the append and the attention one after the other, whoever's context a new row is in."""
import ctypes

import pytest
import torch

from ironcore_amd import _lib, paged_ops, workloads
from ironcore_amd.layers import RotaryPositionalEmbedding

pytestmark = pytest.mark.gpu


def _separately(query, key, value, pools, tables, lens, slots, longest, scale, positions, emb):
    b, _, hn, hd = query.shape
    gn = key.shape[2]
    q = query.reshape(b, hn, hd).clone()
    if emb is None:
        paged_ops.kv_append(key.reshape(b, gn, hd), value.reshape(b, gn, hd), *pools, slots)
    else:
        paged_ops.rope_kv_append(q, key.reshape(b, gn, hd), value.reshape(b, gn, hd), *pools, slots, positions, emb.cos_emb,
                                 emb.sin_emb)
    return paged_ops.paged_decode(q, *pools, tables, lens, longest, scale=scale).view(b, 1, hn * hd)

Call = _lib.STRUCTS["ic_decode_append_call"]


def _together(query, key, value, pools, tables, lens, slots, longest, scale, positions, emb):
    """(return code, output) of the one launch."""
    b, _, hn, hd = query.shape
    n_blocks, gn, block, _ = pools[0].shape
    out = torch.empty(b, 1, hn * hd, dtype=query.dtype, device=query.device)
    call = Call(out=out.data_ptr(), out_stride_seq=hn * hd, q=query.data_ptr(), q_stride_seq=hn * hd, k_new=key.data_ptr(),
                v_new=value.data_ptr(), new_stride_token=key.stride(0), k_pool=pools[0].data_ptr(), v_pool=pools[1].data_ptr(),
                pool_stride_block=pools[0].stride(0), pool_stride_head=pools[0].stride(1), pool_stride_token=pools[0].stride(2),
                num_blocks=n_blocks, block_tables=tables.data_ptr(), block_table_stride=tables.stride(0),
                context_lens=lens.data_ptr(), slot_mapping=slots.data_ptr(), positions=positions.data_ptr(), n_seqs=b, hn=hn,
                gn=gn, hd=hd, block_size=block, max_context_len=longest, scale=scale, dtype=_lib.IC_DTYPE[query.dtype])
    if emb is not None:
        call.cos_table, call.sin_table, call.table_rows = emb.cos_emb.data_ptr(), emb.sin_emb.data_ptr(), emb.cos_emb.shape[0]
    return _lib.load().ic_paged_decode_append(ctypes.byref(call), _lib.current_stream_ptr(query.device)), out


def _by_the_binding(query, key, value, pools, tables, lens, slots, longest, scale, positions, emb):
    angles = (None, None, None) if emb is None else (positions, emb.cos_emb, emb.sin_emb)
    return _lib.host().decode_step(query, key, value, *pools, tables, lens, slots, longest, scale, 1, None, *angles,
                                   *_lib.here(query))


def _compare(gpu, dtype, lens, tables, slots, hn, gn, hd, block, n_blocks, rope, seed, one_launch=True):
    b = len(lens)
    g = torch.Generator(device=gpu).manual_seed(seed)
    pools = [torch.randn(n_blocks, gn, block, hd, generator=g, device=gpu).to(dtype) for _ in range(2)]
    kv = torch.randn(b, 1, 2 * gn * hd, generator=g, device=gpu).to(dtype)
    key, value = (t.view(b, 1, gn, hd) for t in kv.chunk(2, dim=-1))
    query = torch.randn(b, 1, hn, hd, generator=g, device=gpu).to(dtype)
    lens = torch.tensor(lens, dtype=torch.int32, device=gpu)
    positions = torch.randint(-1, 400, (b,), generator=g, device=gpu, dtype=torch.int32)     # clamped into the table
    emb = RotaryPositionalEmbedding(hd, max_seq_len=300).to(gpu) if rope else None
    args = (tables.to(gpu), lens, slots.to(gpu), int(lens.max()), hd ** -0.5, positions, emb)
    apart, mine, bound = ([p.clone() for p in pools] for _ in range(3))
    want = _separately(query, key, value, apart, *args)
    code, got = _together(query, key, value, mine, *args)
    assert code == (0 if one_launch else -3)
    if one_launch:
        assert torch.equal(got, want)
        assert torch.equal(mine[0], apart[0]) and torch.equal(mine[1], apart[1])
    assert torch.equal(_by_the_binding(query, key, value, bound, *args), want)
    assert torch.equal(bound[0], apart[0]) and torch.equal(bound[1], apart[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("hn,gn,hd,block", [(12, 12, 64, 16), (4, 2, 128, 48), (6, 2, 128, 16), (8, 2, 32, 16),
                                            (4, 4, 32, 32)])
@pytest.mark.parametrize("rope", [False, True])
def test_edges(gpu, dtype, hn, gn, hd, block, rope):
    lens = [1, 15, 16, 17, 128, 129, 0, 255, 30]
    wl = workloads.make_decode_workload(len(lens), hn, gn, hd, 255, 255, block_size=block, dtype=dtype, seed=hn)
    last = torch.tensor(lens) - 1
    last[6] = 40                               # an empty context: its row is stored all the same
    slots = wl.block_tables.long().gather(1, (last // block).unsqueeze(1)).squeeze(1) * block + last % block
    slots[8] = -1                              # padding: the last token of row 8 is the pool's
    _compare(gpu, dtype, lens, wl.block_tables, slots, hn, gn, hd, block, wl.k_pool.shape[0], rope, hn + hd)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("hn,gn,hd", [(4, 4, 64), (8, 2, 64)])
def test_rows_that_see_each_other(gpu, dtype, rope, hn, gn, hd):
    """Several new tokens of one sequence as rows of one step; a slot that another row sees in the middle of its
    context; a slot past the pool."""
    block, n_blocks = 16, 12
    table = torch.arange(10, dtype=torch.int32)
    tables = table.repeat(7, 1)
    lens = [61, 62, 63, 64, 65, 150, 150]
    slots = torch.tensor([60, 61, 62, 63, 64, 5, n_blocks * block])
    _compare(gpu, dtype, lens, tables, slots, hn, gn, hd, block, n_blocks, rope, 3)


@pytest.mark.parametrize("b,one", [(64, True), (65, False), (300, False)])
def test_a_row_to_every_lane_and_more(gpu, b, one):
    wl = workloads.make_decode_workload(b, 2, 2, 64, 20, 40, dtype=torch.bfloat16, seed=b)
    last = wl.context_lens.long() - 1
    slots = wl.block_tables.long().gather(1, (last // 16).unsqueeze(1)).squeeze(1) * 16 + last % 16
    tables = wl.block_tables.clone()
    tables[3], slots[3] = tables[b - 1], slots[b - 1] - 1          # row 3 is the last row's sequence, a token earlier
    wl.context_lens[3] = wl.context_lens[b - 1]
    _compare(gpu, torch.bfloat16, wl.context_lens.tolist(), tables, slots, 2, 2, 64, 16, wl.k_pool.shape[0],
             True, b, one_launch=one)


@pytest.mark.parametrize("dtype,hn,gn,hd,b,longest,one", [
    (torch.bfloat16, 4, 4, 128, 3, 1024, True), (torch.bfloat16, 4, 4, 128, 3, 1025, False),      # rounds x head dim
    (torch.float32, 3, 3, 64, 5, 2048, True), (torch.float16, 8, 8, 32, 4, 2047, True),
    (torch.float32, 3, 3, 64, 5, 2049, False),                                                    # the split's
    (torch.bfloat16, 4, 2, 64, 2, 1024, True), (torch.bfloat16, 4, 2, 64, 2, 1025, False),
    (torch.bfloat16, 6, 2, 64, 3, 512, True), (torch.bfloat16, 8, 2, 64, 3, 513, False),
    (torch.bfloat16, 16, 16, 64, 16, 130, True), (torch.bfloat16, 16, 16, 64, 17, 130, False),    # a pair to a CU (256)
    (torch.bfloat16, 8, 4, 64, 64, 256, True), (torch.bfloat16, 8, 4, 64, 64, 257, False),        # pairs x rounds
    (torch.bfloat16, 16, 4, 64, 32, 256, True), (torch.bfloat16, 16, 4, 64, 33, 128, False)])
@pytest.mark.parametrize("rope", [False, True])
def test_rounds_and_the_line_to_two_launches(gpu, dtype, hn, gn, hd, b, longest, one, rope):
    wl = workloads.make_decode_workload(b, hn, gn, hd, longest, longest, dtype=dtype, seed=longest)
    wl.context_lens -= torch.arange(b, dtype=torch.int32)
    wl.context_lens[1] = longest // 2
    last = wl.context_lens.long() - 1
    slots = wl.block_tables.long().gather(1, (last // 16).unsqueeze(1)).squeeze(1) * 16 + last % 16
    tables = wl.block_tables.clone()
    tables[1, :-1] = tables[0, :-1]            # row 1 is in the middle of row 0's context
    slots[1] = tables[1, last[1] // 16].long() * 16 + last[1] % 16
    _compare(gpu, dtype, wl.context_lens.tolist(), tables, slots, hn, gn, hd, 16, wl.k_pool.shape[0], rope, b,
             one_launch=one)
