"""What the step linear refuses on the host, before any launch (no GPU needed)."""
import ctypes

import pytest

from ironcore_amd import _lib
from test_gpu_step_linear import Call

OK = dict(out=1 << 12, out_stride=512, x=1 << 13, x_stride=256, w=1 << 14, w_stride=512, m=4, k=256, n=512)
ROWS = dict(OK, residual=1 << 15, residual_stride=512, norm=1, norm_weight=1 << 16, norm_out=1 << 17, norm_out_stride=512)
APPEND = dict(OK, out_stride=256, n=512, hn=4, gn=2, hd=64, block_size=16, num_blocks=8, k_pool=1 << 15, v_pool=1 << 16,
              pool_stride_block=2048, pool_stride_head=1024, pool_stride_token=64, slot_mapping=1 << 17)


@pytest.mark.parametrize("call,code", [
    (dict(OK, m=-1), -2), (dict(OK, m=33), -3), (dict(OK, n=516), -3), (dict(OK, k=240), -3), (dict(OK, dtype=3), -3),
    (dict(OK, act=6), -3), (dict(OK, tile_bytes=96), -3), (dict(OK, act=5, n=264), -3), (dict(OK, n2=8), -2),
    (dict(OK, act=4, n2=8), -3), (dict(OK, out_stride=504), -2), (dict(OK, x_stride=128), -2), (dict(OK, w=None), -1),
    (dict(OK, x=None), -1), (dict(OK, out=None), -1), (dict(OK, x=(1 << 13) + 8), -6), (dict(OK, out_stride=516), -6),
    (dict(ROWS, act=2), -3), (dict(ROWS, n2=8), -3), (dict(ROWS, norm_out=None), -1), (dict(ROWS, norm_weight=None), -1),
    (dict(ROWS, norm=3), -3), (dict(ROWS, n=16392, w_stride=16392), -3), (dict(ROWS, residual_stride=8), -2), (dict(ROWS), -4),
    (dict(OK, splits=2), -4), (dict(OK, splits=-1), -2),
    (dict(APPEND, act=1), -3), (dict(APPEND, residual=1 << 18), -3), (dict(APPEND, gn=1), -2), (dict(APPEND, k_pool=None), -1),
    (dict(APPEND, cos_table=1 << 18), -1), (dict(APPEND, cos_table=1 << 18, sin_table=1 << 19), -1),
    (dict(APPEND, pool_stride_token=60), -6)])
def test_refused(call, code):
    lib = _lib.load()
    assert lib.ic_step_linear(ctypes.byref(Call(**call)), None) == code


def test_empty_and_sizes():
    lib = _lib.load()
    assert lib.ic_step_linear(None, None) == -1 and lib.ic_step_linear_workspace_bytes(None) == 0
    assert lib.ic_step_linear(ctypes.byref(Call(**dict(OK, m=0))), None) == 0
    assert lib.ic_step_linear(ctypes.byref(Call(**dict(OK, n=0))), None) == 0
    assert lib.ic_step_linear_workspace_bytes(ctypes.byref(Call(**dict(OK, splits=1)))) == 0
    assert lib.ic_step_linear_workspace_bytes(ctypes.byref(Call(**dict(ROWS, splits=1)))) == 4 * 4 * 512
