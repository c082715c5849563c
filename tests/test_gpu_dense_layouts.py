"""Dense calls on tensors that are not laid out row by row: key and value at
strides of their own (an uncached rotary model), heads-first tensors, a query
seen transposed, slices that start at any element, keys shared by a batch.  Each
takes the native call (nothing else may run, and a packed mask is not unpacked)
and returns the bits of the row-major call, which the oracle checks."""
import pytest
import torch

from ironcore_amd import config as ic_config, paged_ops
from ironcore_amd.layers import Attention
from ironcore_amd.layers import attention as attention_module
from oracle.dense_attention import dense_attention
from parity_bars import hold

pytestmark = pytest.mark.gpu

DTYPES = [(torch.bfloat16, "bf16"), (torch.float16, "fp16"), (torch.float32, "fp32")]


def _layer(hn, gn, hd, precision):
    return Attention(ic_config.MainConfig(
        model=ic_config.ModelConfig(d_model=hn * hd, num_attention_heads=hn, num_attention_groups=gn, head_dim=hd,
                                    dropout_attn=0.0, precision=precision),
        trainer=ic_config.TrainerConfig(use_flash_attn=False))).eval()


def _heads_first(t):
    return t.transpose(1, 2).contiguous().transpose(1, 2)


def _half(t):
    """The second half of a projection twice as wide."""
    b, s, h, hd = t.shape
    wide = torch.zeros(b, s, 2 * h * hd, dtype=t.dtype, device=t.device)
    wide[..., h * hd:] = t.reshape(b, s, -1)
    return wide.chunk(2, dim=-1)[1].view(b, s, h, hd)


def _odd_start(t):
    wide = torch.zeros(*t.shape[:3], t.shape[3] + 8, dtype=t.dtype, device=t.device)
    wide[..., 1:t.shape[3] + 1] = t
    return wide[..., 1:t.shape[3] + 1]


LAYOUTS = {
    "rotary": lambda q, k, v: (q, k, _half(v)),
    "halves": lambda q, k, v: (_half(q), _half(k), _half(v)),
    "heads_first": lambda q, k, v: tuple(map(_heads_first, (q, k, v))),
    "query_heads_first": lambda q, k, v: (_heads_first(q), k, v),
    "value_heads_first": lambda q, k, v: (q, k, _heads_first(v)),
    "odd_start": lambda q, k, v: (q, _odd_start(k), _odd_start(v)),
}


def _mask(kind, b, sq, sk, gpu):
    if kind == "none":
        return None
    j, i = torch.arange(sk), torch.arange(sq).unsqueeze(1)
    causal = j <= sk - sq + i
    if kind == "documents":       # a document boundary of its own in each sequence
        cut = torch.tensor([sk // 2 + 3 * n for n in range(b)]).view(b, 1, 1, 1)
        causal = causal & ((j < cut) == (i + sk - sq < cut))
    return causal.expand(b, 1, sq, sk).contiguous().to(gpu) if kind == "documents" else causal.view(1, 1, sq, sk).to(gpu)


@pytest.mark.parametrize("dtype,precision", DTYPES)
@pytest.mark.parametrize("b,sq,sk,hn,gn,hd", [(3, 150, 150, 6, 2, 64), (1, 33, 70, 4, 4, 128), (2, 1, 1, 2, 1, 32)])
@pytest.mark.parametrize("kind", ["none", "causal", "documents"])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_layouts(gpu, monkeypatch, dtype, precision, b, sq, sk, hn, gn, hd, kind, layout):
    g = torch.Generator().manual_seed(sq + sk)
    q, k, v = (torch.randn(b, n, h, hd, generator=g).to(dtype) for n, h in ((sq, hn), (sk, gn), (sk, gn)))
    mask = _mask(kind, b, sq, sk, gpu)
    attn = _layer(hn, gn, hd, precision)

    def fails(*args, **kw):
        raise AssertionError("the call left the native path")
    monkeypatch.setattr(paged_ops, "paged_prefill", fails)
    monkeypatch.setattr(attention_module.PackedMask, "bytes", fails)
    want = attn(q.to(gpu), k.to(gpu), v.to(gpu), mask)
    given = LAYOUTS[layout](q.to(gpu), k.to(gpu), v.to(gpu))
    kept = [t.clone() for t in given]
    assert torch.equal(attn(*given, mask), want)
    assert all(torch.equal(a, b) for a, b in zip(given, kept))
    cpu_mask = None if mask is None else mask.cpu()
    fewest = 1 if mask is not None and sq == sk else sk - sq + 1 if mask is not None else sk
    hold(want, dense_attention(q, k, v, cpu_mask), dense_attention(q.double(), k.double(), v.double(), cpu_mask), dtype,
         fewest, layout)


def test_keys_shared_by_a_batch(gpu):
    """A batch that sees one sequence's keys and values by expand() (no stride between its sequences)."""
    g = torch.Generator(device=gpu).manual_seed(3)
    q = torch.randn(3, 40, 4, 64, generator=g, device=gpu).bfloat16()
    k, v = (torch.randn(1, 40, 2, 64, generator=g, device=gpu).bfloat16().expand(3, 40, 2, 64) for _ in range(2))
    attn, mask = _layer(4, 2, 64, "bf16"), _mask("documents", 3, 40, 40, gpu)
    assert torch.equal(attn(q, k, v, mask), attn(q, k.contiguous(), v.contiguous(), mask))


def test_a_general_mask_costs_no_unpacking(gpu):
    """Memory of a layer call on a mask that is known: the output and the copy of
    the values (4 MiB each), nothing that grows with the mask."""
    b, s, h, hd = 2, 1024, 16, 64
    q, k, v = (torch.randn(b, s, h, hd, device=gpu).bfloat16() for _ in range(3))
    v = _half(v)
    attn, mask = _layer(h, h, hd, "bf16"), _mask("documents", b, s, s, gpu)
    attn(q, k, v, mask)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = attn(q, k, v, mask)
    assert torch.cuda.max_memory_allocated() - before <= 9 << 20 and out.shape == (b, s, h * hd)


def test_unpacking(gpu):
    """What bytes() returns, and the memory it takes: a few bytes for each of the mask's."""
    m = torch.rand(2, 3, 500, 900, device=gpu) < 0.4
    bits, lists, _ = attention_module._lib.host().pack_mask(m.view(torch.uint8), *attention_module._lib.here(m))
    packed = attention_module.PackedMask(bits, lists, tuple(m.shape))
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    got = packed.bytes()
    assert torch.cuda.max_memory_allocated() - before <= 4 * m.numel()
    assert got.dtype == torch.uint8 and torch.equal(got, m.to(torch.uint8))


@pytest.mark.parametrize("dtype,precision", DTYPES)
@pytest.mark.parametrize("hn,gn,hd", [(4, 2, 64), (6, 6, 32), (8, 2, 128)])
@pytest.mark.parametrize("kind", ["none", "documents"])
@pytest.mark.parametrize("layout", ["one_for_all", "odd_distance", "odd_start", "last_of_a_row"])
def test_one_query_row_a_sequence(gpu, dtype, precision, hn, gn, hd, kind, layout):
    """Rows of a query [b, 1, hn, hd] wherever they lie: one for the whole batch (stride 0), at a distance or a start
    that is no multiple of 16 bytes, and at one that is."""
    b, sk = 3, 77
    g = torch.Generator().manual_seed(hn + hd)
    k, v = (torch.randn(b, sk, gn, hd, generator=g).to(dtype) for _ in range(2))
    if layout == "one_for_all":
        q = torch.randn(1, 1, hn, hd, generator=g).to(dtype).to(gpu).expand(b, 1, hn, hd)
    elif layout == "odd_distance":
        q = torch.randn(b, hn * hd + 2, generator=g).to(dtype).to(gpu)[:, :hn * hd].unflatten(1, (1, hn, hd))
    elif layout == "odd_start":
        q = torch.randn(b, hn * hd + 8, generator=g).to(dtype).to(gpu)[:, 1:hn * hd + 1].unflatten(1, (1, hn, hd))
    else:
        q = torch.randn(b, 5, hn, hd, generator=g).to(dtype).to(gpu)[:, -1:]
    mask = _mask(kind, b, 1, sk, gpu)
    got = _layer(hn, gn, hd, precision)(q, k.to(gpu), v.to(gpu), mask)
    cpu_mask = None if mask is None else mask.cpu()
    hold(got, dense_attention(q.cpu(), k, v, cpu_mask),
         dense_attention(q.cpu().double(), k.double(), v.double(), cpu_mask), dtype, 1 if mask is not None else sk, layout)
