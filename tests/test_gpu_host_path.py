"""The native call path (csrc/host_binding.cpp) against the Python one on the
same arguments: same bits, and arguments that are not ordinary left to Python."""
import pytest
import torch

from ironcore_amd import _lib, config as ic_config, paged_ops, workloads
from ironcore_amd.layers import Attention, PagedAttentionMetadata, RotaryPositionalEmbedding

pytestmark = pytest.mark.gpu


def _layer(hn, gn, hd, precision):
    return Attention(ic_config.MainConfig(
        model=ic_config.ModelConfig(d_model=hn * hd, num_attention_heads=hn, num_attention_groups=gn, head_dim=hd,
                                    dropout_attn=0.0, precision=precision),
        trainer=ic_config.TrainerConfig(use_flash_attn=False))).eval()


def _both(monkeypatch, call):
    native = call()
    monkeypatch.setattr(_lib, "here", lambda t: None)
    plain = call()
    monkeypatch.undo()
    return native, plain


@pytest.mark.parametrize("dtype,precision", [(torch.bfloat16, "bf16"), (torch.float32, "fp32")])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("strided", [False, True])
def test_decode_step(gpu, monkeypatch, dtype, precision, rope, strided):
    hn, gn, hd, b = 8, 2, 64, 5
    wl = workloads.make_decode_workload(b, hn, gn, hd, 1, 300, dtype=dtype, seed=3).to(gpu)
    last = wl.context_lens.long() - 1
    slots = wl.block_tables.long().gather(1, (last // 16).unsqueeze(1)).squeeze(1) * 16 + last % 16
    meta = PagedAttentionMetadata(block_tables=wl.block_tables, context_lens=wl.context_lens, slot_mapping=slots,
                                  max_context_len=wl.max_context_len, positions=last.int())
    g = torch.Generator(device=gpu).manual_seed(1)
    kv = torch.randn(b, 1, 2 * gn * hd, generator=g, device=gpu).to(dtype)
    key, value = (t.view(b, 1, gn, hd) for t in kv.chunk(2, dim=-1))     # as the model hands them over
    query = torch.randn(b, 1, hn, hd, generator=g, device=gpu).to(dtype)
    if strided:
        query = torch.stack([query, query], dim=3)[..., 0, :]            # heads apart: Python makes it contiguous
    emb = RotaryPositionalEmbedding(hd, max_seq_len=300).to(gpu) if rope else None
    attn = _layer(hn, gn, hd, precision)
    pools = [(wl.k_pool.clone(), wl.v_pool.clone()) for _ in range(2)]
    left = list(pools)

    def call():
        return attn(query, key, value, kv_cache=left.pop(), attn_metadata=meta, rotary_pos_emb=emb)
    native, plain = _both(monkeypatch, call)
    assert native.shape == plain.shape == (b, 1, hn * hd) and torch.equal(native, plain)
    assert torch.equal(pools[0][0], pools[1][0]) and torch.equal(pools[0][1], pools[1][1])


def test_paged_decode_and_append(gpu, monkeypatch):
    wl = workloads.make_grpo_workload(2, 4, 8, 2, 128, 64, 1, 90, seed=2).to(gpu)
    shared = torch.full((2,), 4, dtype=torch.int32, device=gpu)
    out = torch.empty(8, 8 * 128 + 64, dtype=torch.bfloat16, device=gpu)[:, :8 * 128]     # rows wider apart than long

    def call():
        return paged_ops.paged_decode(wl.query, wl.k_pool, wl.v_pool, wl.block_tables, wl.context_lens,
                                      wl.max_context_len, out=out, cohort_size=4, cohort_shared_blocks=shared).clone()
    native, plain = _both(monkeypatch, call)
    assert torch.equal(native, plain)
    k = torch.randn(3, 2, 128, device=gpu).bfloat16()
    slots = torch.tensor([5, -1, 17], device=gpu)
    pools = [torch.zeros_like(wl.k_pool) for _ in range(4)]
    left = list(pools)
    _both(monkeypatch, lambda: paged_ops.kv_append(k, k, left.pop(), left.pop(), slots))
    assert torch.equal(pools[0], pools[2]) and torch.equal(pools[1], pools[3]) and pools[0].any()


def test_what_is_not_ordinary_is_refused_by_name(gpu):
    wl = workloads.make_decode_workload(2, 4, 2, 64, 20, 40, seed=1).to(gpu)
    args = (wl.k_pool, wl.v_pool, wl.block_tables, wl.context_lens)
    with pytest.raises(TypeError, match="share a dtype"):
        paged_ops.paged_decode(wl.query.float(), *args, wl.max_context_len)
    with pytest.raises(ValueError, match="exceeds what the block table"):
        paged_ops.paged_decode(wl.query, *args, 10_000)
    with pytest.raises(ValueError, match="context_lens"):
        paged_ops.paged_decode(wl.query, *args[:3], wl.context_lens.long(), wl.max_context_len)
    with pytest.raises(_lib.PagedLibraryError):
        paged_ops.paged_decode(wl.query, *args, wl.max_context_len, min_chunk_tokens=24)


def _ragged(gpu, wl, dtype, block, seed):
    """The layer's view of a prefill workload: padded [b, width] tensors and their metadata."""
    b, width = len(wl.chunk_lens), wl.max_chunk_len
    rows = torch.cat([torch.arange(c) + i * width for i, c in enumerate(wl.chunk_lens)])
    slots = torch.full((b * width,), -1, dtype=torch.int64)
    slots[rows] = wl.slot_mapping
    positions = torch.zeros(b * width, dtype=torch.int32)
    positions[rows] = torch.cat([torch.arange(p, p + c) for p, c in zip(wl.prefix_lens, wl.chunk_lens)]).int()
    even = all(c == width for c in wl.chunk_lens)
    meta = PagedAttentionMetadata(
        block_tables=wl.block_tables.to(gpu), context_lens=wl.context_lens.to(gpu), slot_mapping=slots.to(gpu),
        max_context_len=int(wl.context_lens.max()), cu_seqlens_q=None if even else wl.cu_seqlens_q.to(gpu),
        positions=positions.to(gpu), chunk_rows=None if even else rows.to(gpu), max_chunk_len=width)
    g = torch.Generator(device=gpu).manual_seed(seed)

    def rand(heads):
        return torch.randn(b, width, heads, wl.hd, generator=g, device=gpu).to(dtype)
    return meta, rand(wl.hn), rand(wl.gn), rand(wl.gn)


@pytest.mark.parametrize("dtype,precision", [(torch.bfloat16, "bf16"), (torch.float16, "fp16"), (torch.float32, "fp32")])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("hn,gn,hd,prefix,chunks", [
    (6, 2, 64, (0, 90), (1, 70)), (4, 4, 128, (40, 40), (33, 33)), (7, 1, 128, (0, 0), (3, 200)),
    (4, 4, 32, (0, 30), (0, 45)), (8, 8, 128, (1300, 1400), (250, 256))])   # the last: the long kernel's case
def test_prefill_step(gpu, monkeypatch, dtype, precision, rope, hn, gn, hd, prefix, chunks):
    """Padded rows read and written in place, the query rotated inside the
    kernel: the same bits as packing, rotating and scattering around it."""
    n = 20 if prefix[0] > 1000 else 4    # (enough workgroups that long sweeps leave the short kernel)
    wl = workloads.make_prefill_workload(n, hn, gn, hd, *prefix, *chunks, dtype=dtype, seed=hn + hd)
    meta, query, key, value = _ragged(gpu, wl, dtype, 16, 5)
    emb = RotaryPositionalEmbedding(hd, max_seq_len=int(wl.context_lens.max())).to(gpu) if rope else None
    attn = _layer(hn, gn, hd, precision)
    pools = [(wl.k_pool.to(gpu), wl.v_pool.to(gpu)) for _ in range(2)]
    left = list(pools)

    def call():
        return attn(query, key, value, kv_cache=left.pop(), attn_metadata=meta, rotary_pos_emb=emb)
    native, plain = _both(monkeypatch, call)
    assert torch.isfinite(native.float()).all() and torch.equal(native, plain)
    assert torch.equal(pools[0][0], pools[1][0]) and torch.equal(pools[0][1], pools[1][1])


@pytest.mark.parametrize("dtype,precision", [(torch.bfloat16, "bf16"), (torch.float32, "fp32")])
@pytest.mark.parametrize("placement", ["left", "packed", "reversed"])
@pytest.mark.parametrize("hn,gn,hd,prefix,chunks", [(6, 2, 64, (0, 90), (1, 70)), (8, 8, 128, (1300, 1400), (250, 256))])
def test_chunk_rows_anywhere(gpu, monkeypatch, dtype, precision, placement, hn, gn, hd, prefix, chunks):
    """chunk_rows names the rows of the padded tensors that exist, wherever they are: at the ends of
    their sequences' rows (padding on the left), all of them first, or each chunk last row first."""
    n = 20 if prefix[0] > 1000 else 4
    wl = workloads.make_prefill_workload(n, hn, gn, hd, *prefix, *chunks, dtype=dtype, seed=hn + hd)
    meta, query, key, value = _ragged(gpu, wl, dtype, 16, 5)
    width = query.shape[1]
    lens = (wl.cu_seqlens_q[1:] - wl.cu_seqlens_q[:-1]).tolist()
    old = meta.chunk_rows.tolist()
    if placement == "left":
        new = [i * width + width - c + t for i, c in enumerate(lens) for t in range(c)]
    elif placement == "packed":
        new = list(range(len(old)))
    else:
        new = [i * width + c - 1 - t for i, c in enumerate(lens) for t in range(c)]
    slots, positions = torch.full_like(meta.slot_mapping, -1), torch.zeros_like(meta.positions)
    slots[new], positions[new] = meta.slot_mapping[old], meta.positions[old]
    meta.chunk_rows, meta.slot_mapping, meta.positions = torch.tensor(new, device=gpu), slots, positions
    emb = RotaryPositionalEmbedding(hd, max_seq_len=int(wl.context_lens.max())).to(gpu)
    attn = _layer(hn, gn, hd, precision)
    pools = [(wl.k_pool.to(gpu), wl.v_pool.to(gpu)) for _ in range(2)]
    left = list(pools)

    def call():
        return attn(query, key, value, kv_cache=left.pop(), attn_metadata=meta, rotary_pos_emb=emb)
    native, plain = _both(monkeypatch, call)
    padding = torch.ones(n * width, dtype=torch.bool, device=gpu)
    padding[new] = False
    assert torch.isfinite(native.float()).all() and torch.equal(native, plain)
    assert not native.view(n * width, -1)[padding].any()
    assert torch.equal(pools[0][0], pools[1][0]) and torch.equal(pools[0][1], pools[1][1])


@pytest.mark.parametrize("dtype,precision", [(torch.bfloat16, "bf16"), (torch.float32, "fp32")])
@pytest.mark.parametrize("b,s,hn,gn,hd,masked", [(3, 70, 6, 2, 64, True), (1, 1, 4, 4, 128, False), (2, 129, 4, 1, 128, True),
                                                  (70, 5, 2, 2, 32, True), (1, 2304, 2, 2, 128, False)])
def test_dense_call(gpu, monkeypatch, dtype, precision, b, s, hn, gn, hd, masked):
    """Equal sequences without tables, key and value as two halves of one projection."""
    g = torch.Generator(device=gpu).manual_seed(s)
    query = torch.randn(b, s, hn, hd, generator=g, device=gpu).to(dtype)
    kv = torch.randn(b, s, 2 * gn * hd, generator=g, device=gpu).to(dtype)
    key, value = (t.view(b, s, gn, hd) for t in kv.chunk(2, dim=-1))
    mask = torch.ones(1, 1, s, s, device=gpu).tril() if masked else None
    attn = _layer(hn, gn, hd, precision)
    native, plain = _both(monkeypatch, lambda: attn(query, key, value, mask))
    assert torch.equal(native, plain)


def test_out_of_memory_keeps_its_type(gpu):
    """What the allocator raises inside the native call is torch's own exception, as it was from torch.empty."""
    b, pool = 1 << 22, torch.zeros(1, 1, 16, 128, dtype=torch.bfloat16, device=gpu)
    query = torch.zeros(1, 512, 128, dtype=torch.bfloat16, device=gpu).expand(b, 512, 128)     # 512 GiB of output
    tables = torch.zeros(1, 1, dtype=torch.int32, device=gpu).expand(b, 1)
    with pytest.raises(torch.OutOfMemoryError):
        paged_ops.paged_decode(query, pool, pool, tables, torch.ones(b, dtype=torch.int32, device=gpu), 16)


def _failed_hip_call():
    """Leaves a last error in the runtime that the library was linked to, by a call that the host refuses."""
    import ctypes
    with open("/proc/self/maps") as maps:
        path = next(line.split()[-1] for line in maps if "libamdhip64" in line)
    assert ctypes.CDLL(path).hipSetDevice(1 << 20) != 0


def test_a_failed_launch_is_reported(gpu, monkeypatch):
    """A launch error raises, as it does from the Python path, and is not tried away; the next call runs."""
    wl = workloads.make_decode_workload(3, 4, 2, 64, 20, 40, seed=1).to(gpu)
    k = torch.randn(3, 2, 64, device=gpu).bfloat16()
    q, slots = torch.randn(3, 4, 64, device=gpu).bfloat16(), torch.tensor([0, 17, 33], device=gpu)
    meta = PagedAttentionMetadata(block_tables=wl.block_tables, context_lens=wl.context_lens, slot_mapping=slots,
                                  max_context_len=wl.max_context_len)
    attn = _layer(4, 2, 64, "bf16")
    x, w = torch.randn(4, 64, device=gpu), torch.randn(64, 32, device=gpu)
    calls = [lambda: paged_ops.kv_append(k, k, wl.k_pool, wl.v_pool, slots),
             lambda: paged_ops.paged_decode(wl.query, wl.k_pool, wl.v_pool, wl.block_tables, wl.context_lens,
                                            wl.max_context_len),
             lambda: attn(q[:, None], k[:, None], k[:, None], kv_cache=(wl.k_pool, wl.v_pool), attn_metadata=meta),
             lambda: attn(q[None], k[None], k[None]),
             lambda: _lib.host().linear_rows(x, w, w[0], *_lib.here(x))]
    for n, call in enumerate(calls):
        call()                                              # memory for its output is at hand
        torch.cuda.synchronize()
        _failed_hip_call()
        with pytest.raises(_lib.PagedLibraryError) as err:
            call()
        assert err.value.code == -5, n
        call()
        torch.cuda.synchronize()


@pytest.mark.parametrize("why", ["block size", "query start"])
def test_nothing_is_appended_for_a_call_that_is_not_taken(gpu, why):
    """The binding looks for what the attention does not take before it launches the append."""
    hn, gn, hd, bs = 4, 2, 64, 24 if why == "block size" else 16
    pools = torch.zeros(2, 6, gn, bs, hd, dtype=torch.bfloat16, device=gpu)
    k = torch.ones(3, 1, gn, hd, dtype=torch.bfloat16, device=gpu)
    start = 1 if why == "query start" else 0
    q = torch.ones(3 * hn * hd + 1, dtype=torch.bfloat16, device=gpu)[start:start + 3 * hn * hd].view(3, 1, hn, hd)
    tables = torch.arange(6, dtype=torch.int32, device=gpu).view(3, 2)
    lens, slots = torch.full((3,), 5, dtype=torch.int32, device=gpu), torch.arange(3, device=gpu) * 2 * bs
    host, here = _lib.host(), _lib.here(q)
    assert host.decode_step(q, k, k, *pools, tables, lens, slots, 5, 0.125, 1, None, None, None, None, *here) is None
    assert host.prefill_step(q, k, k, *pools, tables, lens, slots, torch.arange(4, dtype=torch.int32, device=gpu), None, 1,
                             0.125, None, None, None, *here) is None
    assert not pools.any()
    meta = PagedAttentionMetadata(block_tables=tables, context_lens=lens, slot_mapping=slots, max_context_len=5)
    with pytest.raises(_lib.PagedLibraryError):     # and the layer refuses it by name, as before
        _layer(hn, gn, hd, "bf16")(q, k, k, kv_cache=tuple(pools), attn_metadata=meta)


def test_metadata_as_the_python_path_takes_it(gpu, monkeypatch):
    """Bounds that are floats, metadata of another class with only the fields a call needs; and chunk rows
    without their bounds, which neither path takes."""
    from types import SimpleNamespace
    hn, gn, hd, b = 4, 2, 64, 4
    attn = _layer(hn, gn, hd, "bf16")
    wl = workloads.make_grpo_workload(2, 2, hn, gn, hd, 64, 1, 90, seed=2).to(gpu)
    last = wl.context_lens.long() - 1
    slots = wl.block_tables.long().gather(1, (last // 16).unsqueeze(1)).squeeze(1) * 16 + last % 16
    shared = torch.full((2,), 4, dtype=torch.int32, device=gpu)
    meta = SimpleNamespace(block_tables=wl.block_tables, context_lens=wl.context_lens, slot_mapping=slots,
                           max_context_len=float(wl.max_context_len), cohort_size=2.0, cohort_shared_blocks=shared)
    k = torch.randn(b, 1, gn, hd, device=gpu).bfloat16()
    q = torch.randn(b, 1, hn, hd, device=gpu).bfloat16()
    native, plain = _both(monkeypatch, lambda: attn(q, k, k, kv_cache=(wl.k_pool, wl.v_pool), attn_metadata=meta))
    assert torch.equal(native, plain)

    wl = workloads.make_prefill_workload(3, hn, gn, hd, 0, 20, 1, 30, seed=4)
    meta, q, k, v = _ragged(gpu, wl, torch.bfloat16, 16, 1)
    pools = wl.k_pool.to(gpu), wl.v_pool.to(gpu)
    fields = {name: getattr(meta, name) for name in ("block_tables", "context_lens", "slot_mapping", "max_context_len",
                                                     "cu_seqlens_q", "chunk_rows")}
    meta = SimpleNamespace(**fields, max_chunk_len=float(meta.max_chunk_len))
    native, plain = _both(monkeypatch, lambda: attn(q, k, v, kv_cache=pools, attn_metadata=meta))
    assert torch.equal(native, plain)
    meta.cu_seqlens_q = None
    with pytest.raises(AttributeError):
        attn(q, k, v, kv_cache=pools, attn_metadata=meta)
