"""The look at a kernel's assembly that the build takes: blocks that spill or reload before the lanes which a branch had switched
off are on again (no compiler needed)."""
import pytest

from ironcore_amd import build

BRANCH = """_Zkernel:                               ; @_Zkernel
; %%bb.0:
\ts_and_saveexec_b64 s[2:3], vcc
\ts_cbranch_execz .LBB0_2
; %%bb.1:
\tglobal_load_dword v1, v[2:3], off
%s.LBB0_2:
%s\ts_or_b64 exec, exec, s[2:3]
%s\ts_endpgm
"""
STORE = "\tscratch_store_dword off, v97, off offset:216 ; 4-byte Folded Spill\n"
LOAD = "\tscratch_load_dword v97, off, off offset:216 ; 4-byte Folded Reload\n"


@pytest.mark.parametrize("inside,before,after,bad", [
    ("", "", STORE, False), (STORE, "", LOAD, False),                    # behind the mask; of the masked lanes' own block
    ("", "\ts_mov_b32 s17, s18\n" + STORE, "", True), ("", LOAD, "", True)])
def test_blocks(inside, before, after, bad):
    assert build.masked_spills(BRANCH % (inside, before, after)) == (["_Zkernel .LBB0_2"] if bad else [])
