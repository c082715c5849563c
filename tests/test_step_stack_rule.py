"""Which steps go to the one launch for all layers: sizes next to each line of the rule, on the side where it was measured
to be the faster way and on the other (no GPU needed)."""
import pytest
import torch

from ironcore_amd import _lib

F, B, H = torch.float32, torch.bfloat16, torch.float16
GELU, SWIGLU = 2, 5


@pytest.mark.parametrize("want,args", [   # type, rows, d, ffn, heads, KV heads, head dim, activation, longest context
    (True, (F, 4, 768, 3072, 12, 12, 64, GELU, 192)), (True, (F, 16, 768, 4096, 12, 12, 64, GELU, 2048)),
    (False, (F, 17, 768, 3072, 12, 12, 64, GELU, 192)), (False, (F, 4, 768, 3072, 12, 12, 64, GELU, 2049)),
    (False, (F, 4, 784, 3072, 12, 12, 64, GELU, 192)), (False, (F, 4, 1024, 4096, 8, 8, 128, GELU, 192)),
    (False, (F, 4, 768, 2304, 6, 6, 128, GELU, 192)),
    (True, (F, 4, 768, 8192, 12, 12, 64, GELU, 192)), (False, (F, 4, 768, 8208, 12, 12, 64, GELU, 192)),
    (False, (F, 5, 768, 4112, 12, 12, 64, GELU, 192)),
    (True, (F, 16, 768, 3072, 12, 4, 64, GELU, 512)), (False, (F, 16, 768, 3072, 12, 4, 64, GELU, 513)),
    (True, (F, 4, 768, 3072, 12, 6, 64, GELU, 192)), (False, (F, 5, 768, 3072, 12, 6, 64, GELU, 192)),
    (False, (F, 4, 256, 352, 4, 4, 64, GELU, 192)),
    (True, (B, 16, 1024, 8192, 8, 8, 128, SWIGLU, 2048)), (False, (B, 16, 1024, 8224, 8, 8, 128, SWIGLU, 2048)),
    (False, (B, 16, 1056, 2752, 8, 8, 128, SWIGLU, 200)), (False, (B, 16, 1024, 2752, 8, 8, 128, SWIGLU, 2049)),
    (True, (H, 16, 1024, 2752, 16, 4, 64, SWIGLU, 512)), (False, (H, 16, 1024, 2752, 16, 4, 64, SWIGLU, 513)),
    (False, (B, 4, 1024, 2752, 16, 2, 64, SWIGLU, 200)), (True, (B, 16, 1024, 2752, 16, 8, 64, SWIGLU, 512)),
    (True, (B, 4, 1024, 2752, 8, 2, 128, SWIGLU, 384)), (False, (B, 5, 1024, 2752, 8, 2, 128, SWIGLU, 384)),
    (False, (B, 4, 1024, 2752, 8, 2, 128, SWIGLU, 385)), (False, (B, 4, 1024, 2752, 8, 4, 128, SWIGLU, 200)),
    (False, (H, 2, 1024, 2752, 8, 2, 128, SWIGLU, 200)),
    (False, (B, 4, 512, 2048, 16, 16, 32, GELU, 200)), (False, (B, 4, 512, 2048, 8, 3, 64, GELU, 200)),
    (False, (B, 0, 1024, 2752, 8, 8, 128, SWIGLU, 200)), (False, (torch.float64, 4, 768, 3072, 12, 12, 64, GELU, 192))])
def test_lines(want, args):
    assert _lib.host().stack_takes(*args) is want
