"""The build's check of the compiled kernels for spills that lose lanes."""
import pytest

from hba_amd.build import lost_spills

# the bf16 query gradient as one build had it: v[16:17] is spilled where the
# loop's exit arrives with no lane on and the branch with those that skipped it
LOST = """
kern:
; %bb.0:
	v_cmp_gt_i32_e32 vcc, s14, v0
	s_and_saveexec_b64 s[8:9], vcc
	s_cbranch_execz .LBB0_310
; %bb.308:
	v_mov_b32_e32 v12, 0
.LBB0_309:                              ; =>This Inner Loop Header: Depth=1
	ds_write_b32 v10, v12
	v_add_u32_e32 v10, 0x1000, v10
	s_andn2_b64 exec, exec, s[10:11]
	s_cbranch_execnz .LBB0_309
.LBB0_310:
	{spill}
	s_or_b64 exec, exec, s[8:9]
	{after}
	s_endpgm
"""


@pytest.mark.parametrize("spill", [
    "scratch_store_dwordx2 off, v[16:17], off offset:40 ; 8-byte Folded Spill",
    "v_accvgpr_write_b32 a212, v0            ;  Reload Reuse",
    "v_mov_b32_e32 v20, v16",
])
def test_vector_instructions_before_the_restore_are_found(spill):
    found = lost_spills(LOST.format(spill=spill, after="s_nop 0"))
    assert [(k, s) for _, k, s in found] == [("kern", spill)]
    assert not lost_spills(LOST.format(spill="s_nop 0", after=spill))   # every lane is on again
    # the loop's exit without the branch's label
    alone = LOST.format(spill=spill, after="s_nop 0").replace(".LBB0_310:", "; %bb.310:")
    assert len(lost_spills(alone)) == 1


def test_spills_at_the_end_of_a_branch_are_found():
    body = "\tscratch_store_dword off, v3, off ; 4-byte Folded Spill\n"
    asm = "kern:\n\ts_and_saveexec_b64 s[0:1], vcc\n\tv_mov_b32_e32 v3, 0\n" + body + "\ts_or_b64 exec, exec, s[0:1]\n"
    assert len(lost_spills(asm)) == 1
    assert not lost_spills(asm.replace(body, ""))          # the branch's own instructions


def test_scalar_spills_are_no_vector_instructions():
    for s in ("v_writelane_b32 v127, s78, 41", "v_readlane_b32 s18, v255, 12", "s_waitcnt lgkmcnt(0)"):
        assert not lost_spills(LOST.format(spill=s, after="s_nop 0"))
