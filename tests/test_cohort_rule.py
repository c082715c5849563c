"""From which sizes on a layer's decode call reads its cohorts' shared blocks once: sizes next to each line of the rule, on the
side where it was measured to be the faster way and on the other (no GPU needed)."""
import pytest

from ironcore_amd import _lib


@pytest.mark.parametrize("want,args", [   # rows, heads, KV heads, head dim, longest context, cohort, bytes of an element
    (False, (64, 12, 12, 128, 488, 16, 2)), (True, (64, 12, 12, 128, 490, 16, 2)),          # 192 MB
    (False, (320, 28, 4, 128, 80, 16, 2)), (False, (320, 28, 4, 128, 80, 1, 2)),
    (True, (160, 28, 4, 64, 612, 16, 2)), (True, (50, 28, 4, 64, 612, 10, 2)),               # grouped heads of 64, many rows
    (False, (160, 28, 4, 64, 612, 8, 2)), (False, (30, 28, 4, 64, 612, 10, 2)),              # 56 columns; 120 pairs
    (True, (48, 28, 4, 64, 952, 16, 2)), (False, (47, 28, 4, 64, 952, 16, 2)),               # 192 pairs
    (True, (32, 64, 8, 64, 612, 16, 2)), (False, (32, 64, 8, 64, 612, 8, 2)),                # 128 columns; 64
    (True, (72, 32, 8, 64, 612, 24, 2)), (False, (64, 32, 8, 64, 612, 32, 2)),               # the pair kernel's 512 pairs
    (True, (48, 16, 4, 64, 1025, 24, 2)), (False, (48, 16, 4, 64, 1024, 24, 2)),             # and its contexts
    (False, (192, 16, 8, 64, 356, 64, 2)),                                                    # two heads to a KV head
    (False, (160, 28, 4, 32, 340, 16, 2)), (False, (160, 28, 4, 128, 340, 16, 2))])           # other head dims
def test_lines(want, args):
    assert _lib.host().cohorts_pay(*args) is want
