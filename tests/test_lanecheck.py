"""The build's check of the compiler's listings (lanecheck.py) on short listings."""
import pytest

from ps3d_amd.lanecheck import misplaced_spills

KERNEL = """
k_pass:                                 ; @k_pass
; %%bb.0:
	v_add_f64 v[116:117], v[2:3], v[4:5]
	s_and_saveexec_b64 s[2:3], s[8:9]
	s_cbranch_execz .LBB0_2
; %%bb.1:
%s
.LBB0_2:
%s
	s_endpgm
.Lfunc_end0:
"""
STORE = "\tscratch_store_dwordx2 off, v[116:117], off offset:16 ; 8-byte Folded Spill"
LOAD = "\tscratch_load_dwordx2 v[116:117], off, off offset:16 ; 8-byte Folded Reload"
KEEP = "\tv_accvgpr_write_b32 a3, v116             ;  Reload Reuse"
ON = "\ts_or_b64 exec, exec, s[2:3]"
WRITE = "\tds_write_b64 v1, v[116:117]"
FORM = "\tv_mul_f64 v[116:117], v[6:7], v[8:9]"


@pytest.mark.parametrize("then, join", [([WRITE], [STORE, ON]), ([WRITE], [LOAD, ON, WRITE]), ([WRITE], [KEEP, ON]),
                                        ([WRITE, STORE, ON], [])])
def test_spills_before_the_lanes_are_restored_are_found(then, join):
    found = misplaced_spills(KERNEL % ("\n".join(then), "\n".join(join)))
    assert [k for k, _ in found] == ["k_pass"]


@pytest.mark.parametrize("then, join", [([WRITE], [ON, STORE, WRITE]), ([WRITE], [ON, LOAD, WRITE]),
                                        ([LOAD, WRITE, ON], []),           # used inside the branch
                                        ([FORM, STORE, ON], [])])          # formed inside the branch
def test_spills_in_their_place_are_not(then, join):
    assert misplaced_spills(KERNEL % ("\n".join(then), "\n".join(join))) == []
