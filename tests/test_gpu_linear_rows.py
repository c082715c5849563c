"""The few-row linear (csrc/linear_rows.hip) at the edges of its tiles: one k
step and many, columns that end inside a tile, splits that do not divide, one
row, a full 16, one more, 32; against float64, and what it leaves to torch."""
import pytest
import torch

from ironcore_amd import _lib, generation

pytestmark = pytest.mark.gpu

# rounding to the element type; fp32: sums of up to 2 816 products in another order
TOL = {torch.bfloat16: 4e-3, torch.float16: 5e-4, torch.float32: 2e-6}


def _operands(gpu, dtype, m, k, n, seed):
    g = torch.Generator().manual_seed(seed)
    x, w, bias = torch.randn(m, k, generator=g), torch.randn(k, n, generator=g) * 0.05, torch.randn(n, generator=g)
    return tuple(t.to(dtype).to(gpu) for t in (x, w, bias))


def _product(x, w, bias, splits=0):
    """The library's entry point itself: none of the binding's rules about what is worth it."""
    lib, dev, (m, k), n = _lib.load(), x.device, x.shape, w.shape[1]
    need = lib.ic_linear_rows_workspace_bytes(m, n, k, splits, _lib.IC_DTYPE[x.dtype])
    ws, out = torch.empty(max(need, 1), dtype=torch.uint8, device=dev), torch.empty(m, n, dtype=x.dtype, device=dev)
    assert lib.ic_linear_rows(out.data_ptr(), n, x.data_ptr(), k, w.data_ptr(), w.stride(0),
                              bias.data_ptr() if bias is not None else None, m, n, k, splits, ws.data_ptr(), need,
                              _lib.IC_DTYPE[x.dtype], _lib.current_stream_ptr(dev)) == 0
    return out


def _distance(got, want):
    return ((got.double().cpu() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,k,n", [(1, 32, 8), (1, 64, 136), (4, 768, 768), (16, 2816, 264), (17, 256, 1000),
                                   (32, 4096, 128), (3, 96, 72)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_against_float64(gpu, dtype, m, k, n, with_bias):
    x, w, bias = _operands(gpu, dtype, m, k, n, m + n)
    def call(w):
        return _lib.host().linear_rows(x, w, bias, *_lib.here(x)) if with_bias else _product(x, w, None)
    got = call(w)
    want = x.double().cpu() @ w.double().cpu()
    if with_bias:
        want = want + bias.double().cpu()
    assert got.shape == (m, n) and got.dtype == dtype
    assert _distance(got, want) <= TOL[dtype]
    wide = torch.zeros(k, n + 8, dtype=dtype, device=gpu)
    wide[:, :n] = w                                     # rows further apart than long: the same sums
    assert torch.equal(call(wide[:, :n]), got)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("splits", [1, 2, 4])
@pytest.mark.parametrize("m", [1, 16, 17, 32])
def test_without_a_bias(gpu, dtype, splits, m):
    """Stored by the products' kernel (one split) and by the sums' (several), one and two blocks of 16 rows."""
    x, w, _ = _operands(gpu, dtype, m, 2080, 200, m + splits)
    want = x.double().cpu() @ w.double().cpu()
    assert _distance(_product(x, w, None, splits), want) <= TOL[dtype]


def test_without_a_bias_through_the_binding(gpu):
    x, w, _ = _operands(gpu, torch.bfloat16, 16, 2048, 256, 3)
    got = _lib.host().linear_rows(x, w, None, *_lib.here(x))
    assert torch.equal(got, _product(x, w, None)) and torch.equal(generation.linear(x, w), got)


@pytest.mark.parametrize("splits", [1, 2, 3, 5])
def test_any_split(gpu, splits):
    x, w, bias = _operands(gpu, torch.float32, 7, 1056, 200, splits)    # 66 steps: splits of unequal length
    lib, dev = _lib.load(), x.device
    need = lib.ic_linear_rows_workspace_bytes(7, 200, 1056, splits, 2)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=dev)
    out = torch.empty(7, 200, device=dev)
    args = (out.data_ptr(), 200, x.data_ptr(), 1056, w.data_ptr(), 200, bias.data_ptr(), 7, 200, 1056, splits)
    assert lib.ic_linear_rows(*args, ws.data_ptr(), need, 2, _lib.current_stream_ptr(dev)) == 0
    want = x.double().cpu() @ w.double().cpu() + bias.double().cpu()
    assert _distance(out, want) <= TOL[torch.float32]
    if need:
        assert lib.ic_linear_rows(*args, ws.data_ptr(), need - 1, 2, _lib.current_stream_ptr(dev)) == -4


def test_what_is_left_to_torch(gpu):
    """Gradients, autocast, vmap and shapes that the kernel does not take go through torch's product."""
    x, w, bias = _operands(gpu, torch.float32, 4, 64, 32, 1)
    want = torch.matmul(x, w) + bias
    host, here = _lib.host(), _lib.here(x)
    wg = w.clone().requires_grad_()
    assert host.linear_rows(x, wg, bias, *here) is None
    generation.linear(x, wg, bias).sum().backward()
    assert torch.allclose(wg.grad, x.sum(0).unsqueeze(1).expand(64, 32), atol=1e-4)
    with torch.no_grad():
        assert host.linear_rows(x, wg, bias, *here) is not None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert torch.matmul(x, w).dtype == torch.bfloat16 and host.linear_rows(x, w, None, *here) is None
        assert torch.allclose(torch.vmap(lambda v: generation.linear(v, w, bias))(x), want, atol=1e-4)
        assert host.linear_rows(x, w, None, *here) is None      # short columns, no bias: torch's is as fast
        for bad in (x[:, ::2], x.double(), torch.zeros(33, 64, device=gpu), torch.zeros(0, 64, device=gpu)):
            assert host.linear_rows(bad, w, bias, *here) is None
        assert host.linear_rows(x, w[:, :30], bias[:30], *here) is None and host.linear_rows(x, w.t(), None, *here) is None
        odd = torch.empty(4 * 64 + 1, device=gpu)[1:].view(4, 64).copy_(x)      # not 16-byte aligned
        assert torch.allclose(generation.linear(odd, w, bias), want, atol=1e-4)


def test_a_bias_that_torch_has_to_see(gpu):
    class Seen(torch.Tensor):
        pass
    x, w, bias = _operands(gpu, torch.float32, 4, 64, 32, 1)
    y = generation.linear(x, w, bias.as_subclass(Seen))
    assert type(y) is Seen and torch.equal(y.as_subclass(torch.Tensor), torch.matmul(x, w) + bias)


F32, BF16 = torch.float32, torch.bfloat16


@pytest.mark.parametrize("dtype,with_bias,m,k,n,taken", [
    (F32, False, 8, 768, 1024, True), (F32, False, 8, 704, 1024, False), (F32, False, 9, 768, 1024, False),
    (F32, False, 9, 1024, 1024, True), (F32, False, 17, 1024, 2048, True), (F32, False, 17, 1024, 4096, False),
    (F32, False, 17, 3072, 4096, True), (F32, False, 4, 2048, 8192, False), (F32, False, 4, 1536, 8192, True),
    (F32, False, 4, 4096, 7168, True), (F32, False, 4, 8192, 8192, True), (F32, False, 16, 1024, 11008, True),
    (F32, False, 17, 1024, 11008, False), (F32, False, 4, 640, 32768, True), (F32, False, 4, 640, 32772, False),
    (F32, True, 32, 512, 2048, True), (F32, True, 16, 1024, 11008, True), (F32, True, 17, 1024, 11008, False),
    (F32, True, 17, 768, 16384, True), (F32, True, 17, 768, 16388, False), (F32, True, 4, 640, 32772, False),
    (F32, True, 4, 2048, 8192, True), (F32, True, 17, 2048, 8192, False), (F32, True, 32, 2048, 4096, True),
    (BF16, False, 16, 2048, 1024, True), (BF16, False, 16, 1792, 1024, False), (BF16, False, 16, 1536, 5120, True),
    (BF16, False, 17, 1536, 5120, False), (BF16, False, 17, 2048, 2048, True), (BF16, False, 4, 4096, 16384, False),
    (BF16, False, 4, 4096, 14336, True), (BF16, False, 4, 8192, 16384, True), (BF16, False, 4, 1088, 16384, True),
    (BF16, False, 4, 2048, 32768, True), (BF16, False, 4, 2048, 32776, False), (BF16, True, 32, 256, 256, True),
    (BF16, True, 4, 2048, 32776, True)])
def test_what_the_library_does_as_fast(gpu, dtype, with_bias, m, k, n, taken):
    """The lines of the rule by size, from both sides (a GPU of 256 CUs)."""
    x, w = torch.zeros(m, k, dtype=dtype, device=gpu), torch.zeros(k, n, dtype=dtype, device=gpu)
    bias = torch.zeros(n, dtype=dtype, device=gpu) if with_bias else None
    y = _lib.host().linear_rows(x, w, bias, *_lib.here(x))
    assert (y is not None) == taken and (not taken or not y.any())
