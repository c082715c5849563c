"""Greedy token choice and a step's bookkeeping (csrc/choose_token.hip) against torch, bit for bit:
chunk edges, ties across chunks, infinities and NaN, finished rows, output columns."""
import pytest
import torch

from ironcore_amd import _lib

pytestmark = pytest.mark.gpu


def _logits(kind, b, n, dtype):
    g = torch.Generator().manual_seed(b + n)
    x = torch.randn(b, n, generator=g).to(dtype)
    rows = torch.arange(b)
    at = torch.randint(0, n, (b, 3), generator=g)
    if kind == "ties":                        # the largest value several times, in other chunks too
        x[rows.unsqueeze(1), at] = 9.0
    elif kind == "nan":
        x[rows.unsqueeze(1), at] = float("nan")
    elif kind == "inf":
        x[rows, at[:, 0]] = float("inf")
        x[0, at[0, 1]] = float("inf")
    elif kind == "lowest":                    # nothing but minus infinity (an argmax there is still the first), one row
        x[0] = float("-inf")
        x[-1, 1:] = float("-inf")
    elif kind == "equal":
        x.fill_(0.0)
        x[:, n // 2] = -0.0
    return x


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", ["plain", "ties", "nan", "inf", "lowest", "equal"])
@pytest.mark.parametrize("b,n", [(1, 8), (3, 4096), (17, 4104), (4, 50304), (33, 12296)])
def test_choice(gpu, dtype, kind, b, n):
    x = _logits(kind, b, n, dtype)
    logits = torch.full((b, n + 8), 99.0, dtype=dtype, device=gpu)[:, :n].copy_(x)    # rows further apart than long
    want = x.argmax(-1, keepdim=True)          # on the CPU: the first of the largest, NaN the largest
    top = torch.topk(x.float(), 2, dim=-1)[0]
    margin = top[:, 0] - top[:, 1]
    tokens = torch.full((b, 5), -7, dtype=torch.int64, device=gpu)
    margins = torch.full((b, 5), -7.0, device=gpu)
    nxt = torch.empty(b, 1, dtype=torch.int64, device=gpu)
    column = torch.tensor([3], device=gpu)
    assert _lib.host().greedy(logits, column, tokens, margins, nxt, None, 0, *_lib.here(logits))
    assert torch.equal(nxt.cpu(), want) and torch.equal(tokens[:, 3:4].cpu(), want)
    assert torch.equal(torch.nan_to_num(margins[:, 3].cpu(), nan=-1.0), torch.nan_to_num(margin, nan=-1.0))
    tokens[:, 3], margins[:, 3] = -7, -7
    column.fill_(5)                            # past the end: not stored
    assert _lib.host().greedy(logits, column, tokens, margins, None, None, 0, *_lib.here(logits))
    assert (tokens == -7).all() and (margins == -7).all()
    done = torch.zeros(b, dtype=torch.bool, device=gpu)
    done[::2] = True
    eos = int(want[-1])
    assert _lib.host().greedy(logits, None, tokens, None, nxt, done, eos, *_lib.here(logits))
    expect = want.clone()
    expect[::2] = eos
    assert torch.equal(nxt.cpu(), expect) and torch.equal(tokens[:, :1].cpu(), expect)
    assert torch.equal(done.cpu(), (torch.arange(b) % 2 == 0) | (expect.squeeze(1) == eos))


def test_what_is_left_to_torch(gpu):
    x = torch.randn(4, 64, device=gpu)
    host, here, nxt = _lib.host(), _lib.here(x), torch.empty(4, 1, dtype=torch.int64, device=gpu)
    for bad in (x.double(), x[:, ::2], x[:, 1:], x[:, :62], x[:0], x.view(2, 2, 64), x.cpu()):
        assert not host.greedy(bad, None, None, None, nxt, None, 0, *here)
    assert not host.greedy(x, None, None, None, nxt.int(), None, 0, *here)
    assert not host.greedy(x, None, nxt.view(2, 2), None, nxt, None, 0, *here)


@pytest.mark.parametrize("b,block", [(1, 16), (5, 48), (300, 16)])
def test_advance(gpu, b, block):
    g = torch.Generator().manual_seed(b)
    tables = torch.randint(0, 1000, (b, 9), generator=g, dtype=torch.int32)[:, :7]
    lens = torch.randint(0, 7 * block, (b,), generator=g, dtype=torch.int32)
    lens[-1] = 7 * block                        # no block left: no slot
    on = lens.to(gpu)
    table = torch.zeros(b, 9, dtype=torch.int32, device=gpu)[:, :7].copy_(tables)
    pos, token_pos = torch.empty_like(on), torch.empty(b, 1, dtype=torch.int64, device=gpu)
    slots, column = torch.empty(b, dtype=torch.int64, device=gpu), torch.tensor([4], device=gpu)
    assert _lib.host().advance(on, table, block, pos, token_pos, slots, column, *_lib.here(on))
    want = tables.long().gather(1, (lens.long() // block).clamp(max=6).unsqueeze(1)).squeeze(1) * block + lens % block
    want[lens >= 7 * block] = -1
    assert torch.equal(on.cpu(), lens + 1) and torch.equal(pos.cpu(), lens) and torch.equal(token_pos.cpu(), lens.long().unsqueeze(1))
    assert torch.equal(slots.cpu(), want) and column.item() == 5
