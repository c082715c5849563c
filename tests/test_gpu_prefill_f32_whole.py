"""The fp32 chunk kernel that gives a wave 32 rows and all keys (csrc/paged_prefill_f32.hip): grids on its side of the line
to the one that splits the keys, short sweeps and long ones, at every head dim; against the same attention in float64."""
import pytest
import torch

from ironcore_amd import paged_ops
from test_gpu_prefill_f32_split import TOL, _attend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("hn,gn,block,seqs", [   # blocks of 32 rows, counted with the longest chunk
    (16, 16, 16, [(i % 7, 1 + 9 * i) for i in range(12)]),                 # 768, contexts up to 106 tokens
    (8, 2, 48, [(0, 144), (10, 129), (79, 65), (3, 128), (0, 1), (80, 64), (16, 127), (1, 33)]),   # 320, up to 144 in wide blocks
    (32, 8, 16, [(300 + i, 97 + i) for i in range(8)]),                    # 1 024, long sweeps
    (28, 4, 80, [(0, 0), (500, 100), (31, 128), (1, 31), (250, 70), (64, 64), (0, 128), (100, 120)])])   # 896, one chunk empty
def test_against_float64(gpu, hd, hn, gn, block, seqs):
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
    longest = max(c for _, c in seqs)
    cells, room = -(-longest // 32) * hn * len(seqs), max(n_blocks) * block
    assert cells > (800 if room > 7 * 32 else 256)
    out = paged_ops.paged_prefill(q.to(gpu), pools[0].to(gpu), pools[1].to(gpu), tables.to(gpu),
                                  torch.tensor(ctx, dtype=torch.int32, device=gpu), cu.to(gpu), longest, scale=hd ** -0.5).cpu()
    for i, (p, c) in enumerate(seqs):
        if c == 0:
            continue
        rows = [pools[j][tables[i, :n_blocks[i]].long()].permute(0, 2, 1, 3).reshape(-1, gn, hd)[:ctx[i]] for j in (0, 1)]
        want = _attend(q[cu[i]:cu[i + 1]], *rows, p, True, hd ** -0.5)
        got = out[cu[i]:cu[i + 1]].view(c, hn, hd).double()
        assert ((got - want).norm() / want.norm()).item() <= TOL, (i, p, c)


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("causal,b,s,heads", [(True, 40, 40, 8), (False, 17, 97, 8), (True, 4, 1100, 16)])
def test_dense(gpu, hd, causal, b, s, heads):
    """(2 240 blocks of 32 rows under the causal rule over long chunks, 544 without a mask, 640 of two tiles.)"""
    from ironcore_amd import config as ic_config
    from ironcore_amd.layers import Attention
    cfg = ic_config.MainConfig(model=ic_config.ModelConfig(d_model=heads * hd, num_attention_heads=heads, num_attention_groups=heads,
                                                           head_dim=hd, dropout_attn=0.0, precision="fp32"),
                               trainer=ic_config.TrainerConfig(use_flash_attn=False))
    layer = Attention(cfg).to(gpu).eval()
    g = torch.Generator().manual_seed(s)
    q, k, v = (torch.randn(b, s, heads, hd, generator=g) for _ in range(3))
    mask = torch.tril(torch.ones(s, s)).view(1, 1, s, s) > 0.5 if causal else None
    with torch.no_grad():
        out = layer(q.to(gpu), k.to(gpu), v.to(gpu), None if mask is None else mask.to(gpu)).cpu().view(b, s, heads, hd)
    for i in {0, b // 2, b - 1}:
        want = _attend(q[i], k[i], v[i], 0, causal, hd ** -0.5)
        assert ((out[i].double() - want).norm() / want.norm()).item() <= 1.5 * TOL   # (longer sums than there)
