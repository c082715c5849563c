"""The layer's decode call with cohorts on both sides of the line from which their shared blocks are read once: the same
result as without cohorts to the rounding of the probabilities, the same pools bit for bit, and cohorts that do not fit refused as ever."""
import numpy as np
import pytest
import torch

from ironcore_amd import config as ic_config
from ironcore_amd.layers import Attention, PagedAttentionMetadata

pytestmark = pytest.mark.gpu


def _call(gpu, dtype, prompts, samples, hn, gn, hd, prefix, own, cohort, shared=None):
    cfg = ic_config.MainConfig(model=ic_config.ModelConfig(d_model=hn * hd, num_attention_heads=hn, num_attention_groups=gn,
                                                           head_dim=hd, dropout_attn=0.0),
                               trainer=ic_config.TrainerConfig(use_flash_attn=False))
    layer = Attention(cfg).to(gpu).eval()
    g = torch.Generator(device=gpu).manual_seed(1)
    b, blocks = prompts * samples, -(-own // 16)
    perm = np.random.default_rng(1).permutation(prompts * (prefix // 16) + b * blocks).astype(np.int32)
    head = np.repeat(perm[:prompts * (prefix // 16)].reshape(prompts, -1), samples, axis=0)
    tables = np.concatenate([head, perm[prompts * (prefix // 16):].reshape(b, blocks)], axis=1)
    ctx = prefix + 1 + np.arange(b) % own
    slots = tables[np.arange(b), (ctx - 1) // 16].astype(np.int64) * 16 + (ctx - 1) % 16
    pools = [torch.randn(len(perm), gn, 16, hd, generator=g, device=gpu).to(dtype) for _ in range(2)]
    q, k, v = (torch.randn(b, 1, n, hd, generator=g, device=gpu).to(dtype) for n in (hn, gn, gn))
    if cohort and shared is None:
        shared = torch.full((prompts,), prefix // 16, dtype=torch.int32, device=gpu)
    meta = PagedAttentionMetadata(
        block_tables=torch.from_numpy(tables).to(gpu), context_lens=torch.from_numpy(ctx.astype(np.int32)).to(gpu),
        slot_mapping=torch.from_numpy(slots).to(gpu), max_context_len=int(ctx.max()), cohort_size=samples if cohort else 1,
        cohort_shared_blocks=shared if cohort else None)
    with torch.no_grad():
        return [layer(q, k, v, None, kv_cache=tuple(pools), attn_metadata=meta), *pools]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(2, 4, 4, 4, 64, 32, 20), (3, 8, 7, 1, 128, 64, 33), (5, 4, 16, 4, 64, 0, 40),
                                   (16, 8, 12, 12, 128, 256, 16), (16, 16, 12, 12, 128, 256, 16)],  # the line: 192 MB
                         ids=lambda s: "-".join(map(str, s)))
def test_as_without_cohorts(gpu, dtype, shape):
    got, want = _call(gpu, dtype, *shape, True), _call(gpu, dtype, *shape, False)
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    # probabilities and the outputs rounded to the type, half a unit of it each, on either side
    off = (got[0].float() - want[0].float()).norm() / want[0].float().norm()
    assert off.item() <= 4 * {torch.bfloat16: 2 ** -9, torch.float16: 2 ** -12}[dtype]


@pytest.mark.parametrize("shape", [(5, 16, 28, 4, 64, 576, 36), (2, 16, 64, 8, 64, 320, 20),   # read once: the line for head dim 64
                                   (2, 16, 28, 4, 64, 576, 36)], ids=lambda s: "-".join(map(str, s)))
def test_many_query_rows_of_head_dim_64(gpu, shape):
    test_as_without_cohorts(gpu, torch.bfloat16, shape)


def test_cohorts_that_do_not_fit_are_refused(gpu):
    with pytest.raises(ValueError):
        _call(gpu, torch.bfloat16, 2, 4, 4, 4, 64, 32, 20, True, torch.zeros(3, dtype=torch.int32, device=gpu))
    with pytest.raises(ValueError):   # 64 members of a cohort are more matrix columns than a workgroup has
        _call(gpu, torch.bfloat16, 1, 64, 16, 1, 64, 32, 20, True)
