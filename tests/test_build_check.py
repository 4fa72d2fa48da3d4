"""The build's look through the device listing for registers that are saved
while lanes are switched off."""
import pytest

from posidonius_amd.build import partial_spills

HEAD = """_Z6kernelv:                             ; @_Z6kernelv
; %bb.0:
	s_and_saveexec_b64 s[2:3], vcc
	s_cbranch_execz .LBB16_41
; %bb.38:
	v_add_f64 v[22:23], v[22:23], v[42:43]
"""
TAIL = """
	v_div_scale_f64 v[22:23], s[2:3], v[14:15], v[14:15], 1.0
	s_endpgm
.Lfunc_end16:
"""
JOIN = ".LBB16_41:                              ;   in Loop: Header=BB16_3 Depth=1\n"
RESTORE = "	s_or_b64 exec, exec, s[2:3]"


@pytest.mark.parametrize("early", [
    "	scratch_store_dwordx2 off, v[106:107], off offset:660 ; 8-byte Folded Spill",
    "	scratch_load_dwordx2 v[106:107], off, off offset:660 ; 8-byte Folded Reload",
    "	v_accvgpr_write_b32 a35, v19",
    "	v_accvgpr_read_b32 v19, a35            ;  Reload Reuse",
    "	v_mov_b64_e32 v[8:9], v[140:141]",
    "	v_mov_b32_e32 v8, v140",
])
def test_registers_saved_before_the_restore_are_found(early):
    listing = HEAD + JOIN + "	s_mov_b32 s23, s35\n" + early + "\n" + RESTORE + TAIL
    found = partial_spills("\t.text\n" + listing + listing.replace("_Z6kernelv", "_Z5otherv"))
    assert found == [f"{k} .LBB16_41: {early.strip()}" for k in ("_Z6kernelv", "_Z5otherv")]


@pytest.mark.parametrize("block", [
    JOIN + "	s_mov_b32 s23, s35\n	v_readlane_b32 s4, v254, 6\n" + RESTORE + "\n	scratch_store_dwordx2 off, v[1:2], off",
    # the tail of the region itself
    "	v_mov_b64_e32 v[8:9], v[140:141]\n" + JOIN + RESTORE,
    # a region that two branches leave early, after arithmetic of its own
    JOIN + "	v_mul_f64 v[4:5], v[90:91], v[178:179]\n	v_mov_b64_e32 v[8:9], v[4:5]\n" + RESTORE,
    # every lane is on, and the next region begins
    JOIN + "	v_mov_b64_e32 v[2:3], v[162:163]\n	s_mov_b64 s[2:3], exec\n	s_mov_b64 exec, s[0:1]",
    # no branch joins here
    JOIN.replace("41", "42") + "	v_mov_b32_e32 v46, v10\n" + RESTORE,
])
def test_ordinary_joins_pass(block):
    assert partial_spills(HEAD + block + TAIL) == []
