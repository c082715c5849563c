"""Append launches whose token rows are narrower than a workgroup, about as wide
and wider: several rows share a workgroup, the last one holds fewer."""
import pytest
import torch

from ironcore_amd import paged_ops
from oracle import paged as oracle_paged
from test_gpu_rope_append import _case, _expect, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hn,gn,hd", [(1, 1, 32), (3, 3, 64), (28, 4, 128), (12, 12, 64), (17, 17, 128)])
@pytest.mark.parametrize("n", [1, 5, 131])
def test_rows_of_any_width(gpu, dtype, hn, gn, hd, n):
    case = _case(n, hn, gn, hd, dtype, seed=n + hd)
    q, k, v, kp, vp, slots, pos, cos, sin = case
    want_q, want_kp, want_vp = _expect(*case)
    qd, kd, vd, kpd, vpd, slotsd, posd, cosd, sind = [t.to(gpu) for t in case]
    paged_ops.rope_kv_append(qd, kd, vd, kpd, vpd, slotsd, posd, cosd, sind)
    assert _same(qd, want_q) and _same(kpd, want_kp) and _same(vpd, want_vp)
    want_k, want_v, skipped = kp.clone(), vp.clone(), slots.clone()
    skipped[n // 2] = -1
    oracle_paged.kv_append(want_k, want_v, k, v, skipped)
    kpd, vpd = kp.to(gpu), vp.to(gpu)
    paged_ops.kv_append(kd, vd, kpd, vpd, skipped.to(gpu))
    assert _same(kpd, want_k) and _same(vpd, want_v)
