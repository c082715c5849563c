"""General masks packed to bits and tile lists (ic_mask_pack) and the dense calls
that read them: the packing against the bytes, and the layer against the byte
path of the same kernels' family and the oracle, at the edges of tiles and query
tiles."""
import pytest
import torch

from ironcore_amd import _lib, config as ic_config, paged_ops
from ironcore_amd.layers import Attention
from ironcore_amd.layers.attention import PackedMask
from oracle.dense_attention import dense_attention
from parity_bars import hold

pytestmark = pytest.mark.gpu


def _mask(n, heads, sq, sk, kind, seed):
    g = torch.Generator().manual_seed(seed)
    if kind == "random":
        m = torch.rand(n, heads, sq, sk, generator=g) < 0.3
    elif kind == "documents":                       # block-diagonal, causal inside a document
        doc = (torch.rand(n, heads, sq, generator=g) < 0.05).cumsum(-1)
        i, j = torch.arange(sq), torch.arange(sk)
        key_doc = torch.nn.functional.pad(doc, (0, max(sk - sq, 0)))[..., :sk]
        m = (doc.unsqueeze(-1) == key_doc.unsqueeze(-2)) & (j <= i.unsqueeze(1))
    else:                                           # a few rows that see nothing among rows that see a far corner
        m = torch.zeros(n, heads, sq, sk, dtype=torch.bool)
        m[..., ::3, -1] = True
    return m


@pytest.mark.parametrize("sq,sk", [(1, 1), (33, 64), (128, 65), (129, 127), (300, 513), (5, 700)])
@pytest.mark.parametrize("kind", ["random", "documents", "corner"])
def test_packing(gpu, sq, sk, kind):
    m = _mask(2, 3, sq, sk, kind, sq + sk)
    wide = torch.zeros(2, 3, sq, sk + 3, dtype=torch.uint8)
    wide[..., 1:sk + 1] = m * 7                     # any nonzero byte is visible; rows start at any byte
    bits, lists, flags = _lib.host().pack_mask(wide.to(gpu)[..., 1:sk + 1], 0, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(PackedMask(bits, lists, tuple(m.shape)).bytes().cpu(), m.to(torch.uint8))
    j, i = torch.arange(sk), torch.arange(sq).unsqueeze(1)
    assert [bool(f) for f in flags.tolist()] == [bool(m.all()), bool((m == (j <= sk - sq + i)).all())]
    lists = lists.cpu().view(6, -1, (sk + 63) // 64 + 1)
    for plane in range(6):
        rows = m.view(6, sq, sk)[plane]
        for qt in range(lists.shape[1]):
            tile_rows = rows[qt * 128:(qt + 1) * 128]
            groups = tile_rows.split(32)
            blind = [bool((~g.any(1)).any()) for g in groups]
            want = []
            for t in range((sk + 63) // 64):
                kinds = [1 if g[:, t * 64:t * 64 + 64].any() or b else 0 for g, b in zip(groups, blind)]
                kinds = [2 if t * 64 + 64 <= sk and g[:, t * 64:t * 64 + 64].all() else k for g, k in zip(groups, kinds)]
                if any(kinds) or any(blind):
                    want.append(t | sum(k << (16 + 2 * n) for n, k in enumerate(kinds)))
            n = int(lists[plane, qt, 0])
            assert lists[plane, qt, 1:1 + n].tolist() == want


@pytest.mark.parametrize("flag,make", [(0, lambda sq, sk: torch.ones(1, 1, sq, sk)),
                                       (1, lambda sq, sk: torch.ones(1, 1, sq, sk).tril(sk - sq))])
@pytest.mark.parametrize("sq,sk", [(1, 2), (64, 64), (70, 133), (129, 129)])
def test_patterns_are_recognised(gpu, flag, make, sq, sk):
    m = make(sq, sk).to(torch.uint8)
    stream = torch.cuda.current_stream().cuda_stream
    flags = _lib.host().pack_mask(m.to(gpu), 0, stream)[2].tolist()
    assert flags[flag] and (sq == 1 or not flags[1 - flag])
    m[0, 0, sq // 2, 0] = 0
    assert _lib.host().pack_mask(m.to(gpu), 0, stream)[2].tolist() == [0, 0]


@pytest.mark.parametrize("dtype,precision", [(torch.bfloat16, "bf16"), (torch.float16, "fp16"), (torch.float32, "fp32")])
@pytest.mark.parametrize("b,sq,sk,hn,gn,hd", [(1, 40, 40, 2, 2, 64), (2, 129, 129, 6, 2, 128), (3, 200, 330, 4, 4, 32),
                                              (2, 300, 70, 2, 1, 64), (20, 260, 260, 8, 8, 64), (1, 70, 700, 3, 1, 128)])
@pytest.mark.parametrize("kind", ["random", "documents", "corner"])
def test_layer(gpu, dtype, precision, b, sq, sk, hn, gn, hd, kind):
    per_seq, per_head = kind != "corner", kind == "random"
    m = _mask(b if per_seq else 1, hn if per_head else 1, sq, sk, kind, sq * 7 + sk)
    g = torch.Generator().manual_seed(sq)
    q, k, v = (torch.randn(b, n, h, hd, generator=g).to(dtype) for n, h in ((sq, hn), (sk, gn), (sk, gn)))
    attn = Attention(ic_config.MainConfig(
        model=ic_config.ModelConfig(d_model=hn * hd, num_attention_heads=hn, num_attention_groups=gn, head_dim=hd,
                                    dropout_attn=0.0, precision=precision),
        trainer=ic_config.TrainerConfig(use_flash_attn=False))).eval()
    out = attn(q.to(gpu), k.to(gpu), v.to(gpu), m.to(gpu))
    ref = dense_attention(q, k, v, m)
    truth = dense_attention(q.double(), k.double(), v.double(), m)
    seen = m.sum(-1)
    fewest = int(torch.where(seen == 0, torch.full_like(seen, sk), seen).min())
    hold(out, ref, truth, dtype, fewest, kind)
    # the byte path of the same call
    pool = (k.to(gpu).permute(0, 2, 1, 3), v.to(gpu).permute(0, 2, 1, 3))
    old = paged_ops.paged_prefill(q.to(gpu).view(b * sq, hn, hd), *pool, torch.arange(b, dtype=torch.int32, device=gpu)[:, None],
                                  torch.full((b,), sk, dtype=torch.int32, device=gpu),
                                  torch.arange(0, (b + 1) * sq, sq, dtype=torch.int32, device=gpu), sq,
                                  mask=m.to(torch.uint8).to(gpu)).view(b, sq, -1)
    bar = {torch.bfloat16: 8e-3, torch.float16: 1e-3, torch.float32: 1e-5}[dtype]   # two roundings of the same sums
    assert ((out - old).abs() <= bar * old.abs().clamp(min=1)).all()


def test_a_mask_given_up_while_another_stream_reads_it(gpu):
    """A mask packed on one stream and used on a second one, then dropped: its packed form is not handed out
    again on the first stream before the second has read it."""
    from ironcore_amd.layers import attention
    n, h, hd = 200, 4, 64
    attn = Attention(ic_config.MainConfig(
        model=ic_config.ModelConfig(d_model=h * hd, num_attention_heads=h, num_attention_groups=h, head_dim=hd,
                                    dropout_attn=0.0, precision="bf16"),
        trainer=ic_config.TrainerConfig(use_flash_attn=False))).eval()
    q = torch.randn(1, n, h, hd, device=gpu).bfloat16()
    mask = _mask(1, 1, n, n, "random", 1).to(gpu)
    want = attn(q, q, q, mask)
    torch.cuda.synchronize()
    packed = attention._MASK_CLASSES[id(mask)][3]
    pieces = [(t.data_ptr(), t.shape, t.dtype) for t in (packed.bits, packed.lists)]
    del packed
    second = torch.cuda.Stream()
    with torch.cuda.stream(second):
        torch.cuda._sleep(50_000_000)
        got = attn(q, q, q, mask)
    del mask                                            # the packed form goes with it
    again = [torch.zeros(shape, dtype=dtype, device=gpu) for _, shape, dtype in pieces]
    assert not {t.data_ptr() for t in again} & {at for at, _, _ in pieces}
    torch.cuda.synchronize()
    assert torch.equal(got, want)
