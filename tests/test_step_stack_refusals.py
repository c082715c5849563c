"""What the call for all layers of a decode step refuses on the host, before any launch (no GPU needed)."""
import ctypes

import pytest

from ironcore_amd import _lib

LAYER = dict(input_norm_weight=1 << 12, q_weight=1 << 13, kv_weight=1 << 14, proj_weight=1 << 15, post_norm_weight=1 << 16,
             up_weight=1 << 17, down_weight=1 << 18, k_pool=1 << 19, v_pool=1 << 20, input_norm=1, post_norm=2,
             input_norm_eps=1e-5, post_norm_eps=1e-5)
OK = dict(x=1 << 12, out=1 << 13, norm_out=1 << 14, norm_weight=1 << 15, num_layers=2, m=4, d=256, f=512, hn=4, gn=2, hd=64, act=2,
          norm=1, eps=1e-5, pool_stride_block=2048, pool_stride_head=1024, pool_stride_token=64, num_blocks=8, block_tables=1 << 16,
          block_table_stride=4, context_lens=1 << 17, slot_mapping=1 << 18, block_size=16, max_context_len=64, scale=0.125,
          dtype=0, workspace=1 << 20, workspace_bytes=1 << 30)


def _call(layer=None, **over):
    lib = _lib.load()
    call = {**OK, **over}
    rows = (_lib.STRUCTS["ic_step_layer"] * 17)(*[_lib.STRUCTS["ic_step_layer"](**LAYER)] * 17)
    for name, value in (layer or {}).items():
        setattr(rows[1], name, value)
    call.setdefault("layers", ctypes.addressof(rows))
    return lib.ic_step_stack(ctypes.byref(_lib.STRUCTS["ic_step_stack_call"](**call)), None)


@pytest.mark.parametrize("over,code", [
    (dict(m=-1), -2), (dict(m=17), -3), (dict(num_layers=-1), -2), (dict(num_layers=17), -3), (dict(d=0), -2), (dict(d=1056), -3),
    (dict(d=248), -3), (dict(f=0), -2), (dict(f=504), -3), (dict(f=(1 << 18) + 32), -3), (dict(hn=5), -3), (dict(hn=10), -3),
    (dict(gn=0), -2), (dict(hd=32), -3), (dict(dtype=3), -3), (dict(dtype=2, d=264), -3), (dict(norm=3), -3), (dict(act=6), -3),
    (dict(block_size=24), -3), (dict(block_size=0), -2), (dict(max_context_len=2049), -3), (dict(max_context_len=65), -2),
    (dict(workgroups=-1), -2), (dict(workgroups=4097), -3), (dict(max_polls=-1), -2), (dict(num_blocks=0), -2),
    (dict(num_blocks=1 << 31), -2), (dict(pool_stride_block=0), -2), (dict(pool_stride_head=-8), -2),
    (dict(pool_stride_token=56), -2),                                    # rows that overlap
    (dict(pool_stride_token=1 << 27), -3), (dict(pool_stride_token=1 << 26, dtype=2), -3),   # past 32 bits in a tile
    (dict(pool_stride_token=68), -6), (dict(pool_stride_head=1028), -6), (dict(pool_stride_block=2052), -6),
    (dict(layers=None), -1), (dict(x=None), -1), (dict(out=None, norm=0), -1), (dict(norm_out=None), -1), (dict(norm_weight=None), -1),
    (dict(block_tables=None), -1), (dict(context_lens=None), -1), (dict(slot_mapping=None), -1), (dict(cos_table=1 << 12), -1),
    (dict(cos_table=1 << 12, sin_table=1 << 13), -1), (dict(cos_table=1 << 12, sin_table=1 << 13, positions=1 << 14), -1),
    (dict(x=(1 << 12) + 8), -6), (dict(out=(1 << 13) + 8), -6), (dict(norm_weight=(1 << 15) + 8), -6),
    (dict(workspace=None), -4), (dict(workspace=(1 << 20) + 128), -4), (dict(workspace_bytes=4096), -4)])
def test_refused(over, code):
    assert _call(**over) == code


@pytest.mark.parametrize("layer,code", [
    ({name: None}, -1) for name in ("input_norm_weight", "q_weight", "kv_weight", "proj_weight", "post_norm_weight", "up_weight",
                                    "down_weight", "k_pool", "v_pool")] + [
    ({"input_norm": 0}, -3), ({"post_norm": 3}, -3), ({"q_bias": 8}, -6), ({"down_weight": (1 << 18) + 8}, -6), ({"v_pool": 8}, -6)])
def test_refused_of_a_layer(layer, code):
    assert _call(layer) == code


def test_empty_and_sizes():
    lib, call = _lib.load(), _lib.STRUCTS["ic_step_stack_call"]
    assert lib.ic_step_stack(None, None) == -1 and lib.ic_step_stack_workspace_bytes(None) == 0
    assert _call(m=0) == 0 and _call(num_layers=0) == 0
    sizes = [lib.ic_step_stack_workspace_bytes(ctypes.byref(call(**{**OK, **over}))) for over in (
        dict(), dict(num_layers=4), dict(m=8), dict(d=1056), dict(m=0))]
    assert 0 < sizes[0] < sizes[1] and sizes[0] < sizes[2] and sizes[3:] == [0, 0]
