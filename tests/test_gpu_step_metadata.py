"""A step's metadata in one upload: the values of the allocator's own lists, the host not waited for in a
model's step, capture refused as before; the prefill's last logits."""
import pytest
import torch

from ironcore_amd import config as ic_config
from ironcore_amd import generation
from ironcore_amd.kv_cache import PagedKVCache

pytestmark = pytest.mark.gpu


def _same(a, b):
    for name in ("block_tables", "context_lens", "slot_mapping", "cu_seqlens_q", "cohort_shared_blocks", "positions", "chunk_rows"):
        x, y = getattr(a, name), getattr(b, name)
        assert (x is None) == (y is None), name
        if x is not None:
            assert x.dtype == y.dtype and torch.equal(x.cpu(), y.cpu()), name
    assert (a.max_context_len, a.cohort_size, a.max_chunk_len) == (b.max_context_len, b.cohort_size, b.max_chunk_len)


def test_prepare_on_the_gpu_and_on_the_cpu(gpu):
    caches = [PagedKVCache(1, 64, 16, 1, 32, torch.float32, dev) for dev in (gpu, "cpu")]
    metas = []
    for cache in caches:
        ids = [cache.add_sequence() for _ in range(3)]
        got = [cache.prepare(ids, [40, 1, 17]), cache.prepare(ids, 1), cache.prepare([], 1), cache.prepare(ids, [0, 3, 0])]
        forks = [ids[0], cache.fork(ids[0]), cache.fork(ids[0]), cache.fork(ids[0])]
        got += [cache.prepare(forks, 1, cohort_size=2), cache.prepare(forks, [16, 2, 33, 1])]
        metas.append(got)
    for a, b in zip(*metas):
        _same(a, b)
    meta = metas[0][0]
    assert meta.positions.is_contiguous() and meta.block_tables.is_contiguous()


def test_slots_a_block_at_a_time():
    """Against one token after the other, aliased blocks included."""
    for counts in ([5], [16], [17], [3, 40, 1], [33]):
        a, b = (PagedKVCache(1, 40, 16, 1, 32, torch.float32, "cpu") for _ in range(2))
        for cache in (a, b):
            root = cache.add_sequence()
            cache.prepare([root], 32)
            cache._seqs[7] = type(cache._seqs[root])(blocks=list(cache._seqs[root].blocks), length=20)    # shares a half-used block
            for blk in cache._seqs[7].blocks:
                cache.allocator.share(blk)
        for c in counts:
            assert a._slots_for_append(a._seqs[7], c) == [b._slot_for_append(b._seqs[7]) for _ in range(c)]
        assert a._seqs[7] == b._seqs[7] and a.allocator._refs == b.allocator._refs


def _model(gpu, dtype, untied):
    cfg = ic_config.MainConfig(
        model=ic_config.ModelConfig(d_model=256, d_ffn=512, num_layers=2, num_attention_heads=4, num_attention_groups=2,
                                    head_dim=64, max_seq_len=96, max_position_embeddings=96, dropout_attn=0.0, dropout_embd=0.0,
                                    dropout_mlp=0.0, untie_embed=untied),
        trainer=ic_config.TrainerConfig(use_flash_attn=False), init=ic_config.InitConfig(seed=0, init_std=0.08))
    torch.manual_seed(0)
    return generation.LanguageModel(cfg, vocab_size=1000).to(gpu).to(dtype).eval()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("untied", [False, True])
@pytest.mark.parametrize("b,lens", [(1, None), (3, None), (3, [5, 21, 1])])
@torch.no_grad()
def test_last_logits_of_a_prefill(gpu, dtype, untied, b, lens):
    model = _model(gpu, dtype, untied)
    ids = torch.randint(0, 1000, (b, 21), generator=torch.Generator().manual_seed(1)).to(gpu)

    def run():
        cache = PagedKVCache(2, 8 * b, 16, 2, 64, dtype, gpu)
        return generation._prefill_logits(model, ids, lens, cache, [cache.add_sequence() for _ in range(b)])
    got = run()
    seen = []
    handle = model.register_forward_hook(lambda *a: seen.append(a[2].shape))
    want = run()                                            # watched: the model is called
    handle.remove()
    assert seen == [(b, 21, model.padded_vocab_size)] and got.shape == want.shape
    tol = 2e-6 if dtype == torch.float32 else 8e-3          # sums of 256 products in other orders; two roundings
    assert ((got.float() - want.float()).norm() / want.float().norm()).item() <= tol


@torch.no_grad()
def test_capture_of_the_bookkeeping_is_refused(gpu):
    model = _model(gpu, torch.float32, False)
    cache = PagedKVCache(2, 8, 16, 2, 64, torch.float32, gpu)
    sid = cache.add_sequence()
    ids = torch.randint(0, 1000, (1, 9)).to(gpu)
    model(ids, kv_cache=cache, seq_ids=[sid])
    before = cache.length(sid), cache.blocks(sid)
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        with pytest.raises(RuntimeError, match="cannot be captured"):
            model(ids[:, :1], kv_cache=cache, seq_ids=[sid])
        ids.add(0)
    assert before == (cache.length(sid), cache.blocks(sid))
    assert torch.isfinite(model(ids[:, :1], kv_cache=cache, seq_ids=[sid])).all()


@torch.no_grad()
def test_under_a_default_device(gpu):
    """The staging memory is the host's, whatever device torch's constructors take by default."""
    model = _model(gpu, torch.float32, False)
    ids = torch.randint(0, 1000, (2, 9), generator=torch.Generator().manual_seed(1)).to(gpu)

    def run():
        cache = PagedKVCache(2, 8, 16, 2, 64, torch.float32, gpu)
        sids = [cache.add_sequence() for _ in range(2)]
        first = model(ids, kv_cache=cache, seq_ids=sids)
        meta = cache.prepare(sids, [3, 1])
        return first, model(ids[:, :1], kv_cache=cache, seq_ids=sids), meta
    want = run()
    with torch.device(gpu):
        got = run()
    _same(got[2], want[2])
    for a, b in zip(got[:2], want[:2]):                     # (under a function mode the modules run, not the native step)
        assert ((a - b).norm() / b.norm()).item() <= 2e-6   # sums of 256 products in other orders


@pytest.mark.parametrize("where", ["instance", "class"])
@torch.no_grad()
def test_a_prepare_of_the_users_own_is_called(gpu, monkeypatch, where):
    model = _model(gpu, torch.float32, False)
    cache = PagedKVCache(2, 8, 16, 2, 64, torch.float32, gpu)
    sid, calls, own = cache.add_sequence(), [], PagedKVCache.prepare

    def prepare(self, seq_ids, new_tokens, *rest):
        calls.append(new_tokens)
        return own(self, seq_ids, new_tokens, *rest)
    if where == "class":
        monkeypatch.setattr(PagedKVCache, "prepare", prepare)
    else:
        cache.prepare = lambda *args: prepare(cache, *args)
    ids = torch.randint(0, 1000, (1, 9)).to(gpu)
    model(ids, kv_cache=cache, seq_ids=[sid])
    model(ids[:, :1], kv_cache=cache, seq_ids=[sid])
    assert calls == [9, 1]


@torch.no_grad()
def test_a_device_without_an_index(gpu, monkeypatch):
    """A cache on "cuda" is on the current GPU, so a model's step does not wait for the upload of its metadata."""
    model = _model(gpu, torch.float32, False)
    cache, waits, upload = PagedKVCache(2, 8, 16, 2, 64, torch.float32, "cuda"), [], PagedKVCache._upload
    monkeypatch.setattr(PagedKVCache, "_upload", lambda self, arrays, wait: (waits.append(wait), upload(self, arrays, wait))[1])
    ids = torch.randint(0, 1000, (1, 9)).to(gpu)
    model(ids, kv_cache=cache, seq_ids=[cache.add_sequence()])
    assert cache.device == cache.k_pools.device == ids.device and waits == [False]
