"""fp32 chunks whose keys are split over the waves of a workgroup (csrc/paged_prefill_f32.hip) at their edges: chunks and
contexts around a tile and a round of tiles, chunks of unequal length, blocks whose tokens lie at one stride and others,
the dense call, head dims, rotary queries; against the oracle in float64."""
import pytest
import torch

from ironcore_amd import paged_ops

pytestmark = pytest.mark.gpu
# fp32 sums of up to 700 products of unit variance: 2^-24 times the square root of their number, with a factor for the exponent
TOL = 4e-6


def _attend(q, k, v, prefix, causal, scale):
    c, hn, _ = q.shape
    g = hn // k.shape[1]
    k, v = (t.double().repeat_interleave(g, 1) for t in (k, v))
    s = torch.einsum("chd,lhd->hcl", q.double(), k) * scale
    if causal:
        hidden = torch.arange(k.shape[0]).unsqueeze(0) > prefix + torch.arange(c).unsqueeze(1)
        s.masked_fill_(hidden, float("-inf"))
    return torch.einsum("hcl,lhd->chd", torch.softmax(s, -1), v)


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("block", [16, 48, 20])
@pytest.mark.parametrize("hn,gn,seqs", [
    (4, 2, [(0, 1)]), (8, 1, [(57, 30)]), (2, 2, [(0, 32), (31, 33), (96, 32), (97, 31)]), (3, 3, [(500, 3), (0, 64), (127, 129)]),
    (4, 4, [(660, 20)])])
def test_against_float64(gpu, hd, block, hn, gn, seqs):
    g = torch.Generator().manual_seed(hd + block)
    ctx = [p + c for p, c in seqs]
    n_blocks = [-(-n // block) for n in ctx]
    perm = torch.randperm(sum(n_blocks), generator=g).to(torch.int32)
    tables = torch.zeros(len(seqs), max(n_blocks), dtype=torch.int32)
    at = 0
    for i, n in enumerate(n_blocks):
        tables[i, :n] = perm[at:at + n]
        at += n
    pools = [torch.randn(sum(n_blocks), gn, block, hd, generator=g) for _ in range(2)]
    q = torch.randn(sum(c for _, c in seqs), hn, hd, generator=g)
    cu = torch.tensor([0] + [c for _, c in seqs], dtype=torch.int32).cumsum(0).to(torch.int32)
    out = paged_ops.paged_prefill(q.to(gpu), pools[0].to(gpu), pools[1].to(gpu), tables.to(gpu),
                                  torch.tensor(ctx, dtype=torch.int32, device=gpu), cu.to(gpu), max(c for _, c in seqs),
                                  scale=hd ** -0.5).cpu()
    for i, (p, c) in enumerate(seqs):
        rows = [pools[j][tables[i, :n_blocks[i]].long()].permute(0, 2, 1, 3).reshape(-1, gn, hd)[:ctx[i]] for j in (0, 1)]
        want = _attend(q[cu[i]:cu[i + 1]], *rows, p, True, hd ** -0.5)
        got = out[cu[i]:cu[i + 1]].view(c, hn, hd).double()
        assert ((got - want).norm() / want.norm()).item() <= TOL, (i, p, c)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("b,s", [(1, 1), (2, 31), (1, 33), (3, 129), (1, 640)])
def test_dense(gpu, hd, causal, b, s):
    from ironcore_amd import config as ic_config
    from ironcore_amd.layers import Attention
    cfg = ic_config.MainConfig(model=ic_config.ModelConfig(d_model=4 * hd, num_attention_heads=4, num_attention_groups=2,
                                                           head_dim=hd, dropout_attn=0.0, precision="fp32"),
                               trainer=ic_config.TrainerConfig(use_flash_attn=False))
    layer = Attention(cfg).to(gpu).eval()
    g = torch.Generator().manual_seed(s)
    q, k, v = (torch.randn(b, s, n, hd, generator=g) for n in (4, 2, 2))
    mask = torch.tril(torch.ones(s, s)).view(1, 1, s, s) > 0.5 if causal else None
    with torch.no_grad():
        out = layer(q.to(gpu), k.to(gpu), v.to(gpu), None if mask is None else mask.to(gpu)).cpu().view(b, s, 4, hd)
    for i in range(b):
        want = _attend(q[i], k[i], v[i], 0, causal, hd ** -0.5)
        assert ((out[i].double() - want).norm() / want.norm()).item() <= TOL


@pytest.mark.parametrize("n,chunk,prefix", [(10, 73, 0), (12, 40, 150), (20, 129, 90)])
def test_a_table_s_room_changes_nothing(gpu, n, chunk, prefix):
    """The layer call knows its longest context: tables with reserved blocks take the same kernel, bit for bit, as
    tables that end with the contexts (more workgroups than CUs, short sweeps: the one that does not split)."""
    from ironcore_amd import config as ic_config
    from ironcore_amd.layers import Attention, PagedAttentionMetadata
    hn, gn, hd = 16, 16, 64
    cfg = ic_config.MainConfig(model=ic_config.ModelConfig(d_model=hn * hd, num_attention_heads=hn, num_attention_groups=gn,
                                                           head_dim=hd, dropout_attn=0.0, precision="fp32"),
                               trainer=ic_config.TrainerConfig(use_flash_attn=False))
    layer = Attention(cfg).to(gpu).eval()
    g = torch.Generator().manual_seed(n)
    blocks = -(-(prefix + chunk) // 16)
    perm = torch.randperm(n * blocks, generator=g).view(n, blocks).to(torch.int32)
    at = torch.arange(prefix, prefix + chunk)
    slots = (perm[:, at // 16].long() * 16 + at % 16).reshape(-1).to(gpu)
    q, k, v = (torch.randn(n, chunk, hn, hd, generator=g).to(gpu) for _ in range(3))
    pools = [torch.randn(n * blocks, gn, 16, hd, generator=g).to(gpu) for _ in range(2)]
    out = []
    for room in (0, 64):
        tables = torch.cat([perm, torch.zeros(n, room, dtype=torch.int32)], dim=1).to(gpu)
        meta = PagedAttentionMetadata(block_tables=tables, slot_mapping=slots, max_context_len=prefix + chunk,
                                      context_lens=torch.full((n,), prefix + chunk, dtype=torch.int32, device=gpu))
        with torch.no_grad():
            out.append(layer(q, k, v, None, kv_cache=tuple(t.clone() for t in pools), attn_metadata=meta))
    assert torch.equal(*out)
