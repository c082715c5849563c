"""Which native calls an eager decode step makes, by its sizes: what a call would refuse for them is neither gathered nor
asked, and the step's numbers are the modules' either way."""
import pytest
import torch

from ironcore_amd import _lib, generation
from ironcore_amd import config as ic_config
from ironcore_amd.kv_cache import PagedKVCache

pytestmark = pytest.mark.gpu


def _model(gpu, d, hn, gn, dtype=torch.bfloat16):
    cfg = ic_config.MainConfig(
        model=ic_config.ModelConfig(d_model=d, d_ffn=2 * d, num_layers=2, num_attention_heads=hn, num_attention_groups=gn,
                                    head_dim=d // hn, max_seq_len=64, max_position_embeddings=64, dropout_attn=0.0,
                                    dropout_embd=0.0, dropout_mlp=0.0, precision="bf16"),
        trainer=ic_config.TrainerConfig(use_flash_attn=False), init=ic_config.InitConfig(seed=0, init_std=0.02))
    torch.manual_seed(1)
    return generation.LanguageModel(cfg, vocab_size=256).to(gpu).to(dtype).eval()


def _step(gpu, model, rows, monkeypatch):
    """(logits, pools) of one decode step and the names of the native calls it made for the layers."""
    cfg, calls, host = model.config.model, [], _lib.host()

    class Counting:
        def __getattr__(self, name):
            if name in ("decoder_stack", "decoder_layer", "norm_rows"):
                calls.append(name)
            return getattr(host, name)
    cache = PagedKVCache(cfg.num_layers, rows, 16, cfg.num_attention_groups, cfg.d_model // cfg.num_attention_heads,
                         model.embedding.word_embeddings.weight.dtype, gpu)
    ids = torch.arange(rows * 4, device=gpu).view(rows, 4) % 250
    with torch.no_grad():
        seqs = [cache.add_sequence() for _ in range(rows)]
        model(ids[:, :3], kv_cache=cache, seq_ids=seqs)
        with monkeypatch.context() as m:
            m.setattr(_lib, "host", lambda proxy=Counting(): proxy)
            out = model(ids[:, 3:], kv_cache=cache, seq_ids=seqs)
    return out, cache, calls


@pytest.mark.parametrize("rows,d,hn,gn,want", [
    (16, 1024, 8, 8, ["decoder_stack"]),                                                    # the stack's largest
    (17, 1024, 8, 8, ["norm_rows", "decoder_layer", "decoder_layer"]),                     # a row more
    (4, 1088, 17, 17, ["norm_rows", "decoder_layer", "decoder_layer"]),                    # wider
    (4, 1024, 16, 2, ["norm_rows", "decoder_layer", "decoder_layer"]),                     # more heads to a KV head
    (4, 512, 16, 16, ["norm_rows", "decoder_layer", "decoder_layer"]),                     # heads of 32
    (33, 512, 8, 8, [])])                                                                   # more rows than any call takes
def test_calls_of_a_step(gpu, monkeypatch, rows, d, hn, gn, want):
    model = _model(gpu, d, hn, gn)
    plans = []
    real = generation._step_plan
    monkeypatch.setattr(generation, "_step_plan", lambda *a: plans.append(1) or real(*a))
    out, cache, calls = _step(gpu, model, rows, monkeypatch)
    assert calls == want and len(plans) == bool(want)
    monkeypatch.setattr(generation, "_step_plan", lambda *a: None)
    modules, other, _ = _step(gpu, model, rows, monkeypatch)
    # two layers of some ten roundings to eight bits on either side
    assert ((out.float() - modules.float()).norm() / modules.float().norm()).item() < 2 * 10 * 2 ** -9
    for a, b in ((cache.k_pools, other.k_pools), (cache.v_pools, other.v_pools)):
        assert ((a.float() - b.float()).norm() / b.float().norm()).item() < 2 * 10 * 2 ** -9
