"""The linears of a decode step with their surroundings (csrc/step_linear.hip): every
form against float64 at the edges of tiles, steps and splits; the native step of a model
against its modules; what is left to the modules."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from ironcore_amd import _lib, generation
from ironcore_amd import config as ic_config
from ironcore_amd.kv_cache import PagedKVCache

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16, torch.float32]
# one rounding to the element type (2^-9, 2^-12; the norm takes a rounded row: two); fp32: sums of 2 080 products
TOL = {torch.bfloat16: 5e-3, torch.float16: 6e-4, torch.float32: 1e-6}

Call = _lib.STRUCTS["ic_step_linear_call"]


def _run(gpu, call, dtype):
    lib = _lib.load()
    call.dtype = _lib.IC_DTYPE[dtype]
    need = lib.ic_step_linear_workspace_bytes(ctypes.byref(call))
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=gpu)
    call.workspace, call.workspace_bytes = ws.data_ptr(), need
    assert lib.ic_step_linear(ctypes.byref(call), _lib.current_stream_ptr(gpu)) == 0
    if need:
        call.workspace_bytes = need - 1
        assert lib.ic_step_linear(ctypes.byref(call), _lib.current_stream_ptr(gpu)) == -4


def _ptr(t):
    return None if t is None else t.data_ptr()


def _distance(got, want):
    return ((got.double().cpu() - want).norm() / want.norm()).item()


def _linear_call(x, w, bias, w2=None, bias2=None, **more):
    return Call(x=x.data_ptr(), x_stride=x.stride(0), w=w.data_ptr(), bias=_ptr(bias), w_stride=w.stride(0), w2=_ptr(w2),
                bias2=_ptr(bias2), w2_stride=w2.stride(0) if w2 is not None else 0, m=x.shape[0], k=x.shape[1],
                n=w.shape[1], n2=w2.shape[1] if w2 is not None else 0, **more)


def _draw(gpu, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return lambda *shape, scale=1.0: (torch.randn(*shape, generator=g) * scale).to(dtype).to(gpu)


SIZES = [(1, 32, 8), (4, 768, 776), (16, 1024, 264), (17, 256, 200), (32, 1056, 520), (5, 2080, 64)]
PLANS = [(0, 0), (64, 1), (64, 3), (128, 1), (128, 8), (256, 1), (256, 9)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tile,splits", PLANS)
@pytest.mark.parametrize("m,k,n", SIZES)
def test_activations(gpu, dtype, tile, splits, m, k, n):
    rand = _draw(gpu, dtype, m + n)
    x = rand(m, k)
    for act, fn in ((0, lambda y: y), (1, F.relu), (2, F.gelu), (3, F.silu),
                    (4, lambda y: y.chunk(2, 1)[0] * y.chunk(2, 1)[1].sigmoid()),
                    (5, lambda y: F.silu(y.chunk(2, 1)[0]) * y.chunk(2, 1)[1])):
        w, bias = rand(k, n * (2 if act > 3 else 1), scale=k ** -0.5), rand(n * (2 if act > 3 else 1))
        w2, bias2 = (rand(k, 72, scale=k ** -0.5), rand(72)) if act < 4 and m > 1 else (None, None)
        cols = n + (72 if w2 is not None else 0)
        out = torch.full((m, cols), float("nan"), dtype=dtype, device=gpu)
        _run(gpu, _linear_call(x, w, bias, w2, bias2, out=out.data_ptr(), out_stride=cols, act=act, tile_bytes=tile,
                               splits=splits), dtype)
        y = x.double().cpu() @ w.double().cpu() + bias.double().cpu()
        if w2 is not None:
            y = torch.cat([y, x.double().cpu() @ w2.double().cpu() + bias2.double().cpu()], 1)
        assert _distance(out, fn(y)) <= TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tile,splits", PLANS)
@pytest.mark.parametrize("m,k,n", SIZES + [(2, 64, 8200)])
def test_residual_and_norm(gpu, dtype, tile, splits, m, k, n):
    rand = _draw(gpu, dtype, m + n)
    x, w, bias, res, gain, shift = rand(m, k), rand(k, n, scale=k ** -0.5), rand(n), rand(m, n) + 2, rand(n), rand(n)
    want = x.double().cpu() @ w.double().cpu() + bias.double().cpu()
    for norm, with_residual in ((0, True), (1, True), (2, True), (1, False)):
        out, normed = (torch.full((m, n), float("nan"), dtype=dtype, device=gpu) for _ in range(2))
        _run(gpu, _linear_call(x, w, bias, out=out.data_ptr(), norm_out=normed.data_ptr(), out_stride=n,
                               norm_out_stride=n, residual=_ptr(res if with_residual else None), residual_stride=n,
                               norm=norm, eps=1e-5, norm_weight=gain.data_ptr(), norm_bias=_ptr(shift if norm == 1 else None),
                               tile_bytes=tile, splits=splits), dtype)
        h = want + res.double().cpu() if with_residual else want
        assert _distance(out, h) <= TOL[dtype]
        h = out.double().cpu()       # the norm takes the row as it was rounded
        if norm == 1:
            h = F.layer_norm(h, (n,), gain.double().cpu(), shift.double().cpu(), 1e-5)
        elif norm == 2:
            h = F.rms_norm(h, (n,), gain.double().cpu(), 1e-5)
        if norm:
            assert _distance(normed, h) <= TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tile,splits", PLANS)
@pytest.mark.parametrize("b,hn,gn,hd,d", [(1, 2, 1, 32, 64), (17, 4, 2, 64, 224), (5, 6, 6, 64, 1056)])
@pytest.mark.parametrize("rope", [False, True])
def test_append(gpu, dtype, tile, splits, b, hn, gn, hd, d, rope):
    rand = _draw(gpu, dtype, b + d)
    x, wq, wkv = rand(b, d), rand(d, hn * hd, scale=d ** -0.5), rand(d, 2 * gn * hd, scale=d ** -0.5)
    bq, bkv = rand(hn * hd), rand(2 * gn * hd)
    pools = [torch.full((5, gn, 16, hd), 7.0, dtype=dtype, device=gpu) for _ in range(2)]
    g = torch.Generator().manual_seed(b)
    slots = torch.randperm(80, generator=g)[:b]
    slots[b // 2] = -1 if b > 1 else slots[b // 2]
    positions = torch.randint(0, 50, (b,), generator=g, dtype=torch.int32)
    angle = torch.randn(50, hd // 2, generator=g) * 3
    cos, sin = angle.cos().to(gpu), angle.sin().to(gpu)
    out = torch.empty(b, hn * hd, dtype=dtype, device=gpu)
    on_gpu, pos_gpu = slots.to(gpu), positions.to(gpu)
    _run(gpu, _linear_call(x, wq, bq, wkv, bkv, out=out.data_ptr(), out_stride=hn * hd, tile_bytes=tile, splits=splits,
                           k_pool=pools[0].data_ptr(), v_pool=pools[1].data_ptr(), pool_stride_block=pools[0].stride(0),
                           pool_stride_head=pools[0].stride(1), pool_stride_token=pools[0].stride(2), num_blocks=5, hn=hn,
                           gn=gn, hd=hd, block_size=16, slot_mapping=on_gpu.data_ptr(), positions=pos_gpu.data_ptr(),
                           cos_table=_ptr(cos if rope else None), sin_table=_ptr(sin if rope else None), table_rows=50), dtype)
    q = (x.double().cpu() @ wq.double().cpu() + bq.double().cpu()).view(b, hn, hd)
    kv = (x.double().cpu() @ wkv.double().cpu() + bkv.double().cpu()).view(b, 2, gn, hd)
    k, v = kv[:, 0], kv[:, 1]
    if rope:
        c, s = (t.double().cpu()[positions.long()].unsqueeze(1) for t in (cos, sin))

        def turn(t):
            return torch.stack([t[..., ::2] * c - t[..., 1::2] * s, t[..., ::2] * s + t[..., 1::2] * c], -1).flatten(-2)
        q, k = turn(q), turn(k)
    assert _distance(out, q.reshape(b, -1)) <= TOL[dtype]
    for pool, rows in zip(pools, (k, v)):
        got = pool.permute(0, 2, 1, 3).reshape(80, gn, hd).cpu()
        there = slots >= 0
        assert _distance(got[slots[there]], rows[there]) <= TOL[dtype]
        untouched = torch.ones(80, dtype=torch.bool)
        untouched[slots[there]] = False
        assert (got[untouched] == 7).all()


def _model(gpu, dtype, vocab=512, **over):
    precision = {torch.bfloat16: "bf16", torch.float16: "fp16", torch.float32: "fp32"}[dtype]
    m = dict(d_model=256, d_ffn=352, num_layers=3, num_attention_heads=4, num_attention_groups=2, head_dim=64,
             max_seq_len=128, max_position_embeddings=128, dropout_attn=0.0, dropout_embd=0.0, dropout_mlp=0.0,
             precision=precision)
    positional = over.pop("positional", "absolute")
    cfg = ic_config.MainConfig(model=ic_config.ModelConfig(**{**m, **over}),
                               trainer=ic_config.TrainerConfig(use_flash_attn=False),
                               init=ic_config.InitConfig(seed=0, init_std=0.08))
    cfg.model.positional_embedding.type = positional
    torch.manual_seed(1)
    model = generation.LanguageModel(cfg, vocab_size=vocab)
    for name, p in model.named_parameters():
        if "bias" in name or "norm" in name:
            p.data += 0.1 * torch.randn(p.shape)
    return model.to(gpu).to(dtype).eval()


@torch.no_grad()
def _steps(model, gpu, b, steps=3):
    """Logits of a prefill and of some steps, and the pools."""
    m = model.config.model
    hd = m.d_model // m.num_attention_heads
    cache = PagedKVCache(m.num_layers, 6 * b, 16, m.num_attention_groups, hd, next(model.parameters()).dtype, gpu)
    sids = [cache.add_sequence() for _ in range(b)]
    ids = torch.randint(0, 500, (b, 21 + steps), generator=torch.Generator().manual_seed(b)).to(gpu)
    logits = [model(ids[:, :21], kv_cache=cache, seq_ids=sids)[:, -1]]
    logits += [model(ids[:, 21 + i:22 + i], kv_cache=cache, seq_ids=sids)[:, -1] for i in range(steps)]
    return torch.stack(logits[1:]).float(), cache.k_pools.float(), cache.v_pools.float()


def _taken(monkeypatch):
    """How many layers ran natively."""
    count = []
    host = _lib.host()

    class Counting:
        def __getattr__(self, name):
            fn = getattr(host, name)
            if name != "decoder_layer":
                return fn

            def call(*a):
                got = fn(*a)
                count.append(got is not None)
                return got
            return call
    monkeypatch.setattr(_lib, "host", lambda proxy=Counting(): proxy)
    return count


def _by_modules(monkeypatch, call):
    with monkeypatch.context() as m:
        m.setattr(generation, "_step_plan", lambda *a: None)
        return call()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("over", [
    dict(), dict(no_bias=True, ln_type="rmsnorm", activation_type="swiglu", positional="rope", untie_embed=True),
    dict(post_ln=True, activation_type="relu", num_attention_groups=1), dict(activation_type="glu", ln_type="rmsnorm"),
    dict(activation_type="silu", num_attention_heads=8, head_dim=32, num_attention_groups=8, positional="rope")])
@pytest.mark.parametrize("b", [1, 17])
def test_model_step(gpu, monkeypatch, dtype, over, b):
    """The native step against the modules: the same to rounding, and no further from the fp32 model."""
    model = _model(gpu, dtype, **over)
    modules = _by_modules(monkeypatch, lambda: _steps(model, gpu, b))
    count = _taken(monkeypatch)
    native = _steps(model, gpu, b)
    assert count == [True] * 9
    exact = _by_modules(monkeypatch, lambda: _steps(_widened(model, gpu, over), gpu, b))
    for got, want, true in zip(native, modules, exact):
        def off(t):
            return ((t - true).norm() / true.norm()).item()
        if dtype == torch.float32:
            assert ((got - want).norm() / want.norm()).item() <= 5e-6   # sums of up to 352 products in other orders, 3 layers
        else:
            assert off(got) <= 1.15 * off(want) + 1e-4                  # two random roundings: within 15 % of each other


def _widened(model, gpu, over):
    wide = _model(gpu, torch.float32, **dict(over))
    wide.load_state_dict({k: v.float() for k, v in model.state_dict().items()})
    return wide


def test_modules_that_are_watched_are_called(gpu, monkeypatch):
    model = _model(gpu, torch.float32)
    want = _steps(model, gpu, 2)
    count = _taken(monkeypatch)
    layer = model.model.layers[1]
    watched = [model.model, layer, layer.input_layernorm, layer.input_layernorm.layernorm, layer.linear_kv, layer.self_attention,
               layer.attn_output, layer.post_attn_layernorm, layer.mlp, layer.mlp.up_proj, layer.mlp.activation,
               layer.mlp.down_proj, model.output_layernorm]
    for module in watched:
        seen = []
        handle = module.register_forward_hook(lambda *a: seen.append(1) and None)
        got = _steps(model, gpu, 2)
        handle.remove()
        assert len(seen) == 4 and not count, type(module)     # the prefill and three steps
        for a, b in zip(got, want):
            assert torch.allclose(a, b, atol=1e-4)
    handle = torch.nn.modules.module.register_module_forward_pre_hook(lambda *a: None)
    _steps(model, gpu, 2)
    handle.remove()
    layer.mlp.forward = lambda x, f=layer.mlp.forward: f(x)
    _steps(model, gpu, 2)
    del layer.mlp.forward
    with monkeypatch.context() as m:
        m.setattr(generation.Linear, "forward", lambda self, x: generation.linear(x, self.weight, self.bias))
        _steps(model, gpu, 2)
    assert not count
    _steps(model, gpu, 2)
    assert count == [True] * 9


def test_what_is_left_to_the_modules(gpu, monkeypatch):
    count = _taken(monkeypatch)
    for over, b in ((dict(activation_type="geglu", d_ffn=256), 2), (dict(), 33)):
        _steps(_model(gpu, torch.float32, **over), gpu, b, steps=1)
        assert not any(count)
        del count[:]
    model = _model(gpu, torch.float32)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        _steps(model, gpu, 2, steps=1)
    assert not any(count)
    # a layer whose weights do not lie as the kernel reads them runs as a module between two native ones
    want = _steps(model, gpu, 2)
    del count[:]
    up = model.model.layers[1].mlp.up_proj
    up.weight.data = up.weight.data.t().contiguous().t()
    got = _steps(model, gpu, 2)
    assert count == [True, False, True] * 3
    for a, b in zip(got, want):
        assert torch.allclose(a, b, atol=1e-4)


def test_step_in_a_graph_and_on_another_stream(gpu):
    model = _model(gpu, torch.bfloat16, positional="rope")
    ids = torch.randint(0, 500, (3, 20), generator=torch.Generator().manual_seed(1)).to(gpu)
    want = generation.generate(model, ids, 12)
    assert torch.equal(generation.generate(model, ids, 12, use_graph=True), want)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        got = generation.generate(model, ids, 12)
    torch.cuda.current_stream().wait_stream(stream)
    assert torch.equal(got, want)
