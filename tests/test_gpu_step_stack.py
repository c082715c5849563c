"""All layers of a decode step in one launch (csrc/step_stack.hip) against the same step in float64.

Sizes: rows of one to the largest number of steps, short last splits of a column, the row counts around the two forms of
the fp32 product, grouped heads, contexts of one tile to several rounds; the work dealt in turn, by fewer workgroups than
CUs, and from the counter, as when other work keeps the workgroups from starting together."""
import ctypes
import math

import pytest
import torch

from ironcore_amd import _lib

pytestmark = pytest.mark.gpu
# Rounded to the element type where the outputs of a layer's parts are (six times a layer): half a unit in the last place
# each, 2^-9, 2^-12 and 2^-25 relative, and as much again for the fp32 sums of up to 4 096 terms; two layers.
TOL = {torch.bfloat16: 2 * 6 * 2 ** -9, torch.float16: 2 * 6 * 2 ** -12, torch.float32: 2e-6}
NORM_LAYER, NORM_RMS = 1, 2
RELU, GELU, SILU, GLU, SWIGLU = 1, 2, 3, 4, 5


def _norm(x, kind, weight, bias, eps):
    if kind == NORM_LAYER:
        x = x - x.mean(-1, keepdim=True)
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight
    return x if bias is None else x + bias


def _act(x, act):
    if act == RELU:
        return x.relu()
    if act == GELU:
        return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))
    if act == SILU:
        return x * torch.sigmoid(x)
    a, b = x.chunk(2, -1)
    return a * torch.sigmoid(b) if act == GLU else a * torch.sigmoid(a) * b


def _turn(x, cos, sin):  # [m, heads, hd], [m, 1, hd / 2]
    a, b = x[..., ::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _oracle(c, layers, x, pools):
    """(last norm's output, pools) in float64."""
    m, hn, gn, hd, bs = c["m"], c["hn"], c["gn"], c["hd"], c["block"]
    for w, (kp, vp) in zip(layers, pools):
        n = _norm(x, c["norm"], w["n1"], w["n1b"], 1e-5)
        q = (n @ w["q"] + w["qb"]).view(m, hn, hd)
        k, v = (n @ w["kv"] + w["kvb"]).view(m, 2, gn, hd).unbind(1)
        if c["rope"]:
            cos, sin = (t.double().cpu()[c["positions"].long()].unsqueeze(1) for t in (c["cos"], c["sin"]))
            q, k = _turn(q, cos, sin), _turn(k, cos, sin)
        for i, slot in enumerate(c["slots"].tolist()):
            if slot >= 0:
                kp[slot // bs, :, slot % bs], vp[slot // bs, :, slot % bs] = k[i], v[i]
        att = torch.zeros(m, hn, hd, dtype=torch.float64)
        for i, ctx in enumerate(c["ctx"]):
            if ctx == 0:
                continue
            blocks = c["tables"][i, :(ctx + bs - 1) // bs].long()
            kk = kp[blocks].permute(0, 2, 1, 3).reshape(-1, gn, hd)[:ctx].repeat_interleave(hn // gn, 1)
            vv = vp[blocks].permute(0, 2, 1, 3).reshape(-1, gn, hd)[:ctx].repeat_interleave(hn // gn, 1)
            p = torch.softmax(torch.einsum("hd,thd->ht", q[i], kk) * c["scale"], -1)
            att[i] = torch.einsum("ht,thd->hd", p, vv)
        x = x + att.reshape(m, -1) @ w["o"] + w["ob"]
        n = _norm(x, c["norm"], w["n2"], w["n2b"], 1e-6)
        x = x + _act(n @ w["up"] + w["upb"], c["act"]) @ w["down"] + w["downb"]
    return x, _norm(x, c["norm"], c["last"].double().cpu(), None, 1e-5)


def _case(gpu, dtype, m, d, f, hn, gn, hd, act, norm, rope, contexts, seed=0, layers=2, block=16):
    g = torch.Generator().manual_seed(seed)

    def rand(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(dtype)
    up = 2 * f if act >= GLU else f
    weights = []
    for _ in range(layers):
        w = {"q": rand(d, hn * hd, std=d ** -0.5), "kv": rand(d, 2 * gn * hd, std=d ** -0.5),
             "o": rand(hn * hd, d, std=(hn * hd) ** -0.5), "up": rand(d, up, std=d ** -0.5), "down": rand(f, d, std=f ** -0.5)}
        w.update(n1=1 + rand(d, std=0.1), n2=1 + rand(d, std=0.1), qb=rand(hn * hd, std=0.1), kvb=rand(2 * gn * hd, std=0.1),
                 ob=rand(d, std=0.1), upb=rand(up, std=0.1), downb=rand(d, std=0.1), n1b=None, n2b=None)
        if norm == NORM_LAYER:
            w.update(n1b=rand(d, std=0.1), n2b=rand(d, std=0.1))
        weights.append(w)
    held = [(c + block - 1) // block for c in contexts]
    n_blocks = sum(held) + 1
    perm = torch.randperm(n_blocks, generator=g).tolist()
    tables = torch.zeros(m, max(held) + 1, dtype=torch.int32)
    slots = []
    for i, c in enumerate(contexts):
        for j in range(held[i]):
            tables[i, j] = perm.pop()
        slots.append(int(tables[i, (c - 1) // block]) * block + (c - 1) % block if c > 0 else -1)
    angles = torch.rand(max(contexts) + 1, hd // 2, generator=g) * 6
    c = {"m": m, "d": d, "f": f, "hn": hn, "gn": gn, "hd": hd, "act": act, "norm": norm, "rope": rope, "ctx": list(contexts),
         "tables": tables, "slots": torch.tensor(slots), "positions": torch.tensor([max(n - 1, 0) for n in contexts], dtype=torch.int32),
         "cos": angles.cos().to(gpu), "sin": angles.sin().to(gpu), "scale": hd ** -0.5, "block": block, "last": (1 + rand(d, std=0.1)).to(gpu)}
    x = rand(m, d)
    pools = [(rand(n_blocks, gn, block, hd), rand(n_blocks, gn, block, hd)) for _ in range(layers)]
    return c, weights, x, pools


def _run(gpu, dtype, c, weights, x, pools, tokens_first=False, **over):
    """(out, norm_out, pools) of the library's call; ``tokens_first``: a block's tokens are its outer rows in the pools."""
    lib = _lib.load()
    keep = [{k: None if t is None else t.to(gpu) for k, t in w.items()} for w in weights]
    on = [tuple(t.to(gpu) for t in kv) for kv in pools]
    if tokens_first:
        on = [tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in kv) for kv in on]
    table = (_lib.STRUCTS["ic_step_layer"] * len(weights))()
    ptr = lambda t: None if t is None else t.data_ptr()
    for row, w, (k, v) in zip(table, keep, on):
        for field, key in (("input_norm_weight", "n1"), ("input_norm_bias", "n1b"), ("q_weight", "q"), ("q_bias", "qb"),
                           ("kv_weight", "kv"), ("kv_bias", "kvb"), ("proj_weight", "o"), ("proj_bias", "ob"),
                           ("post_norm_weight", "n2"), ("post_norm_bias", "n2b"), ("up_weight", "up"), ("up_bias", "upb"),
                           ("down_weight", "down"), ("down_bias", "downb")):
            setattr(row, field, ptr(w[key]))
        row.k_pool, row.v_pool = k.data_ptr(), v.data_ptr()
        row.input_norm = row.post_norm = c["norm"]
        row.input_norm_eps, row.post_norm_eps = 1e-5, 1e-6
    x = x.to(gpu)
    out, norm_out = torch.empty_like(x), torch.empty_like(x)
    meta = [c["tables"].to(gpu), torch.tensor(c["ctx"], dtype=torch.int32, device=gpu), c["slots"].to(gpu), c["positions"].to(gpu)]
    pool = on[0][0]
    call = _lib.STRUCTS["ic_step_stack_call"](
        layers=ctypes.addressof(table), x=x.data_ptr(), out=out.data_ptr(), norm_out=norm_out.data_ptr(),
        norm_weight=c["last"].data_ptr(), num_layers=len(weights), m=c["m"], d=c["d"], f=c["f"], hn=c["hn"], gn=c["gn"], hd=c["hd"],
        act=c["act"], norm=c["norm"], eps=1e-5, pool_stride_block=pool.stride(0), pool_stride_head=pool.stride(1),
        pool_stride_token=pool.stride(2), num_blocks=pool.shape[0], block_tables=meta[0].data_ptr(),
        block_table_stride=meta[0].stride(0), context_lens=meta[1].data_ptr(), slot_mapping=meta[2].data_ptr(),
        positions=meta[3].data_ptr() if c["rope"] else None, cos_table=c["cos"].data_ptr() if c["rope"] else None,
        sin_table=c["sin"].data_ptr() if c["rope"] else None, table_rows=c["cos"].shape[0], block_size=c["block"],
        max_context_len=max(c["ctx"]), scale=c["scale"], dtype=_lib.dtype_code(dtype), **over)
    need = lib.ic_step_stack_workspace_bytes(ctypes.byref(call))
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    call.workspace, call.workspace_bytes = ws.data_ptr(), need
    _lib.check("ic_step_stack", lib.ic_step_stack(ctypes.byref(call), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return out, norm_out, on


def _close(got, want, tol):
    got = got.double().cpu()
    return ((got - want).norm() / want.norm()).item() <= tol


SHAPES = [  # m, d, f, hn, gn, hd, act, norm, rope, contexts
    (1, 64, 64, 1, 1, 64, GELU, NORM_LAYER, False, (1,)),
    (4, 768, 3072, 12, 12, 64, GELU, NORM_LAYER, False, (160, 17, 16, 129)),
    (5, 1024, 2752, 8, 8, 128, SWIGLU, NORM_RMS, True, (33, 300, 1, 128, 48)),
    (16, 512, 1088, 8, 2, 64, GLU, NORM_LAYER, True, tuple(7 + 19 * i for i in range(16))),
    (3, 832, 1344, 13, 13, 64, RELU, NORM_RMS, False, (500, 0, 260)),
    (9, 1024, 1024, 8, 4, 128, SILU, NORM_LAYER, True, tuple(100 + i for i in range(9))),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s[:6])))
def test_against_float64(gpu, dtype, shape):
    c, weights, x, pools = _case(gpu, dtype, *shape)
    wide = [(k.double(), v.double()) for k, v in pools]
    want = _oracle(c, [{k: None if t is None else t.double() for k, t in w.items()} for w in weights], x.double(), wide)
    first = None
    # in turn; with fewer workgroups than CUs; from the counter: the same bits each time
    for over in (dict(), dict(workgroups=37), dict(draw=1), dict(workgroups=5, draw=1)):
        out, normed, after = _run(gpu, dtype, c, weights, x, pools, **over)
        for got, true in zip((out, normed), want):
            assert _close(got, true, TOL[dtype]), over
        for pair, true in zip(after, wide):
            for got, t in zip(pair, true):
                assert _close(got, t, TOL[dtype]), over
        if first is None:
            first = (out, normed)
        assert torch.equal(out, first[0]) and torch.equal(normed, first[1]), over


MORE = [  # m, d, f, hn, gn, hd, act, norm, rope, contexts; block size
    ((4, 256, 512, 16, 16, 64, GELU, NORM_LAYER, False, (200, 3, 64, 31)), 32),      # an output projection in parts (fp32)
    ((3, 512, 576, 16, 16, 128, SWIGLU, NORM_RMS, True, (40, 129, 16)), 48),         # ... and in 16 bits
    ((7, 768, 1024, 12, 4, 64, SILU, NORM_LAYER, True, (511, 512, 513, 128, 127, 1, 257)), 64),   # three heads to a KV head
    ((2, 384, 384, 6, 2, 64, RELU, NORM_RMS, False, (96, 97)), 16),
    ((3, 512, 512, 8, 8, 64, GELU, NORM_LAYER, True, (1024, 2047, 2048)), 16),       # up to 16 tiles a wave
    ((16, 128, 128, 2, 2, 64, GLU, NORM_LAYER, False, (2048,) * 8 + tuple(1900 + 17 * i for i in range(8))), 48),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape,block", MORE, ids=lambda v: "-".join(map(str, v[:6])) if isinstance(v, tuple) else str(v))
def test_projections_groups_blocks_and_long_contexts(gpu, dtype, shape, block):
    c, weights, x, pools = _case(gpu, dtype, *shape, block=block)
    wide = [(k.double(), v.double()) for k, v in pools]
    want = _oracle(c, [{k: None if t is None else t.double() for k, t in w.items()} for w in weights], x.double(), wide)
    first = None
    for over in (dict(), dict(tokens_first=True), dict(draw=1, workgroups=61)):
        out, normed, after = _run(gpu, dtype, c, weights, x, pools, **over)
        for got, true in zip((out, normed), want):
            assert _close(got, true, TOL[dtype]), over
        for pair, true in zip(after, wide):
            for got, t in zip(pair, true):
                assert _close(got, t, TOL[dtype]), over
        first = first or (out, normed)
        assert torch.equal(out, first[0]) and torch.equal(normed, first[1]), over


@pytest.mark.parametrize("m", [4, 5, 16])   # the two forms of the product
def test_fp32_rounds_no_more_than_the_layers_own_launches(gpu, m):
    """Distance to float64 of the last norm, over four draws: not above that of a call per layer."""
    host, off, dtype = _lib.host(), [0.0, 0.0], torch.float32
    for seed in range(4):
        c, weights, x, pools = _case(gpu, dtype, m, 768, 3072, 12, 12, 64, GELU, NORM_LAYER, False,
                                     tuple(60 + 11 * i for i in range(m)), seed=seed)
        wide = [(k.double(), v.double()) for k, v in pools]
        want = _oracle(c, [{k: None if t is None else t.double() for k, t in w.items()} for w in weights], x.double(), wide)[1]
        _, normed, _ = _run(gpu, dtype, c, weights, x, pools)
        w = [{k: None if t is None else t.to(gpu) for k, t in layer.items()} for layer in weights]
        hidden = x.to(gpu).view(m, 1, 768)
        here = _lib.here(hidden)
        n = host.norm_rows(hidden, w[0]["n1"], w[0]["n1b"], NORM_LAYER, 1e-5, *here)
        meta = (c["tables"].to(gpu), torch.tensor(c["ctx"], dtype=torch.int32, device=gpu), c["slots"].to(gpu), max(c["ctx"]))
        for i, layer in enumerate(w):
            after = (w[i + 1]["n1"], w[i + 1]["n1b"]) if i + 1 < len(w) else (c["last"], None)
            hidden, n = host.decoder_layer(
                hidden, n, [layer[k] for k in ("q", "qb", "kv", "kvb", "o", "ob", "n2", "n2b", "up", "upb", "down", "downb")] + [*after],
                12, 12, 64, GELU, NORM_LAYER, 1e-6, NORM_LAYER, 1e-5, False, *(t.to(gpu) for t in pools[i]), *meta, c["scale"], 1,
                None, None, None, None, *here)
        for j, got in enumerate((normed, n.view(m, 768))):
            off[j] += ((got.double().cpu() - want).norm() / want.norm()).item()
    assert off[0] <= off[1]


def test_rows_that_see_each_other(gpu):
    """Two tokens of one sequence as rows of a step, and blocks that two rows share."""
    c, weights, x, pools = _case(gpu, torch.float32, 4, 128, 256, 2, 2, 64, GELU, NORM_LAYER, False, (40, 40, 17, 17))
    c["tables"][1] = c["tables"][0]
    c["tables"][3] = c["tables"][2]
    c["ctx"][0] = 39
    c["slots"][0] = int(c["tables"][0, 2]) * 16 + 38 % 16
    c["slots"][1] = int(c["tables"][0, 2]) * 16 + 39 % 16
    c["slots"][2], c["slots"][3] = int(c["tables"][2, 1]) * 16, -1
    wide = [(k.double(), v.double()) for k, v in pools]
    want = _oracle(c, [{k: None if t is None else t.double() for k, t in w.items()} for w in weights], x.double(), wide)
    out, normed, _ = _run(gpu, torch.float32, c, weights, x, pools)
    assert _close(out, want[0], 2e-6) and _close(normed, want[1], 2e-6)


def test_nan_and_infinity_pass_through(gpu):
    """A row of NaN and one with infinities end as NaN, the others untouched by them; no wait is caught by the value."""
    c, weights, x, pools = _case(gpu, torch.float32, 4, 128, 256, 2, 2, 64, GELU, NORM_LAYER, False, (20, 20, 20, 20))
    clean, _, _ = _run(gpu, torch.float32, c, weights, x, pools)
    x = x.clone()
    x.view(torch.int32)[1] = -1   # every bit set
    x[2, 5] = float("inf")
    out, _, _ = _run(gpu, torch.float32, c, weights, x, pools)
    assert out[1].isnan().all() and out[2].isnan().all()
    assert torch.equal(out[0], clean[0]) and torch.equal(out[3], clean[3])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m", [4, 5])
def test_infinite_weights(gpu, dtype, m):
    """Infinities in the last row of a matrix whose rows do not fill a task's steps: infinite keys where they belong."""
    c, weights, x, pools = _case(gpu, dtype, m, 512, 512, 8, 8, 64, GELU, NORM_LAYER, False, tuple(range(17, 17 + m)), layers=1)
    weights[0]["kv"][511, 3] = float("inf")
    weights[0]["kv"][511, 70] = -float("inf")
    _, _, [(keys, _)] = _run(gpu, dtype, c, weights, x, pools)
    last = _norm(x.double(), NORM_LAYER, weights[0]["n1"].double(), weights[0]["n1b"].double(), 1e-5)[:, 511]
    for i, slot in enumerate(c["slots"].tolist()):
        row = keys[slot // 16, :, slot % 16].cpu().float()
        assert row[0, 3] == float("inf") * last[i].sign() and row[1, 6] == -float("inf") * last[i].sign()
        assert row.isfinite().sum() == row.numel() - 2


@pytest.mark.parametrize("over", [dict(), dict(workgroups=37), dict(draw=1)], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[2], SHAPES[3]], ids=lambda s: "-".join(map(str, s[:6])))
def test_a_wait_that_is_given_up(gpu, dtype, shape, over):
    """With one poll to a wait the launch ends, says so, and appends nothing that is wrong: outputs are the right ones or
    NaN, the pools' rows the right ones or the old ones."""
    c, weights, x, pools = _case(gpu, dtype, *shape)
    out, normed, after = _run(gpu, dtype, c, weights, x, pools, **over)
    status = torch.zeros(1, dtype=torch.int32, device=gpu)
    _run(gpu, dtype, c, weights, x, pools, status=status.data_ptr(), **over)
    assert status.item() == 0
    lost_out, lost_normed, lost_after = _run(gpu, dtype, c, weights, x, pools, status=status.data_ptr(), max_polls=1, **over)
    assert status.item() == 1
    for got, want in ((lost_out, out), (lost_normed, normed)):
        assert got.isnan().any() and bool((got.isnan() | (got == want)).all())
    assert bool((lost_normed.isnan().all(1) | (lost_normed == normed).all(1)).all())
    for pair, right, before in zip(lost_after, after, pools):
        for got, want, old in zip(pair, right, before):
            assert bool(((got == want) | (got == old.to(gpu))).all())


def _model(gpu, dtype, layers):
    from ironcore_amd import config as ic_config
    from ironcore_amd import generation
    cfg = ic_config.MainConfig(
        model=ic_config.ModelConfig(d_model=512, d_ffn=1024, num_layers=layers, num_attention_heads=8, num_attention_groups=8,
                                    head_dim=64, max_seq_len=128, max_position_embeddings=128, dropout_attn=0.0,
                                    dropout_embd=0.0, dropout_mlp=0.0,
                                    precision={torch.float32: "fp32", torch.bfloat16: "bf16"}[dtype]),
        trainer=ic_config.TrainerConfig(use_flash_attn=False), init=ic_config.InitConfig(seed=0, init_std=0.05))
    cfg.model.positional_embedding.type = "rope"
    torch.manual_seed(1)
    return generation.LanguageModel(cfg, vocab_size=512).to(gpu).to(dtype).eval()


def test_model_of_two_parts_two_streams_and_a_graph(gpu, monkeypatch):
    """More layers than one call holds; the step on two streams at once, whose workgroups cannot all be resident together,
    and as a graph: the tokens of the modules."""
    import threading

    from ironcore_amd import generation
    model = _model(gpu, torch.float32, 20)
    ids = torch.randint(0, 500, (3, 20), generator=torch.Generator().manual_seed(1)).to(gpu)
    with monkeypatch.context() as m:
        m.setattr(generation, "_step_plan", lambda *a: None)
        want = generation.generate(model, ids, 24)
    calls = []
    host = _lib.host()

    class Counting:
        def __getattr__(self, name):
            fn = getattr(host, name)
            if name != "decoder_stack":
                return fn
            return lambda *a: calls.append(fn(*a)) or calls[-1]
    monkeypatch.setattr(_lib, "host", lambda proxy=Counting(): proxy)
    assert torch.equal(generation.generate(model, ids, 24), want)
    assert len(calls) == 23 and all(t is not None for t in calls)
    del calls[:]
    assert torch.equal(generation.generate(model, ids, 24, use_graph=True), want)
    got = [None, None]

    def work(i):
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(stream):
            got[i] = generation.generate(model, ids, 24)
        stream.synchronize()
    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert torch.equal(got[0], want) and torch.equal(got[1], want)


def test_a_step_that_gave_up_is_raised(gpu):
    """The next step of the process raises what an earlier one's launch has left in the status word, once."""
    from ironcore_amd import generation
    model = _model(gpu, torch.float32, 2)
    ids = torch.randint(0, 500, (3, 20), generator=torch.Generator().manual_seed(1)).to(gpu)
    want = generation.generate(model, ids, 4)
    torch.cuda.synchronize()
    ctypes.c_int32.from_address(_lib.load().ic_step_status()).value = 1
    with pytest.raises(_lib.PagedLibraryError, match="gave up"):
        generation.generate(model, ids, 4)
    assert torch.equal(generation.generate(model, ids, 4, eos_token_id=511), want)
