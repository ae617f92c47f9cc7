"""The check of what stands around inline assembly, on assembly with one mistake each."""
import pytest

from cacti_amd import asm_check

GOOD = """
kernel:
; %bb.0:
	s_load_dwordx2 s[2:3], s[0:1], 0x0
	v_readfirstlane_b32 s6, v9
	v_mov_b32_e32 v10, 0
	v_accvgpr_write_b32 a0, 0
	v_accvgpr_write_b32 a3, 0
	s_waitcnt lgkmcnt(0)
	s_nop 1
.LBB0_1:                                ; =>This Inner Loop Header: Depth=1
	ds_read_b128 v[4:7], v10 offset:64
	s_waitcnt lgkmcnt(0)
	;;#ASMSTART
	s_add_u32 m0, s6, 0x400
	v_mfma_f32_16x16x32_f16 a[0:3], v[4:7], v[12:15], a[0:3]
	global_load_lds_dwordx4 v8, s[2:3]
	;;#ASMEND
	s_add_i32 s7, s7, 1
	s_cmp_lg_u32 s7, s8
	s_cbranch_scc1 .LBB0_1
; %bb.2:
	;;#ASMSTART
	s_nop 15
	s_nop 15
	;;#ASMEND
	v_accvgpr_read_b32 v16, a3
	v_mul_f32_e32 v16, s9, v16
	v_cvt_f16_f32_e32 v16, v16
	global_store_short v[18:19], v16, off
	s_endpgm
.Lfunc_end0:
	.size	kernel, .Lfunc_end0-kernel
; ScratchSize: 0
"""

MISTAKES = [
    ("the accumulators are copied inside the loop", "\ts_add_i32 s7, s7, 1\n", "\tv_accvgpr_read_b32 v20, a1\n\ts_add_i32 s7, s7, 1\n",
     "touched too early"),
    ("and written at the loop's head, behind the jump", "\tds_read_b128", "\tv_accvgpr_write_b32 a2, v20\n\tds_read_b128", "touched too early"),
    ("stored as they are", "\tv_accvgpr_read_b32 v16, a3\n", "\tglobal_store_dwordx4 v[18:19], a[0:3], off\n", None),
    ("too short a wait", "\ts_nop 15\n\ts_nop 15\n", "\ts_nop 7\n", "touched too early"),
    ("no wait, results stored as they are", "\ts_nop 15\n\ts_nop 15\n\t;;#ASMEND\n\tv_accvgpr_read_b32 v16, a3\n",
     "\t;;#ASMEND\n\tglobal_store_dwordx4 v[18:19], a[0:3], off\n", "touched too early"),
    ("a fragment is moved in front of its product", "\t;;#ASMSTART\n\ts_add_u32 m0", "\tv_mov_b32_e32 v13, v21\n\t;;#ASMSTART\n\ts_add_u32 m0",
     "reads a vector result too early"),
    ("the base comes out of a vector register", "\tds_read_b128 v[4:7], v10 offset:64\n", "\tds_read_b128 v[4:7], v10 offset:64\n\tv_readfirstlane_b32 s3, v22\n",
     "reads a scalar register too early"),
    ("nothing between an address and its load", "\tv_mfma_f32_16x16x32_f16 a[0:3], v[4:7], v[12:15], a[0:3]\n\tglobal_load", "\tglobal_load",
     "follows its address too early"),
    ("the compiler's own M0", "\ts_add_i32 s7, s7, 1\n", "\ts_mov_b32 m0, s7\n\ts_add_i32 s7, s7, 1\n", "uses M0 as well"),
    ("spills", "; ScratchSize: 0", "; ScratchSize: 48", "48 bytes of registers in memory"),
    ("rounded once", "\tv_mul_f32_e32 v16, s9, v16\n\tv_cvt_f16_f32_e32 v16, v16\n", "\tv_fma_mixlo_f16 v16, v16, s9, 0\n", "rounded once"),
]


def test_good_assembly_has_no_faults():
    assert asm_check.check(GOOD) == []


@pytest.mark.parametrize("what,old,new,text", MISTAKES, ids=[m[0].replace(" ", "_") for m in MISTAKES])
def test_one_mistake_is_found(what, old, new, text):
    assert GOOD.count(old) == 1
    faults = asm_check.check(GOOD.replace(old, new))
    if text is None:                                      # not a mistake: behind both waits
        assert faults == []
    else:
        assert faults and text in faults[0], faults


def test_kernels_that_hold_more_registers_than_they_may():
    text = GOOD + "\t.amdhsa_kernel kernel\n\t\t.amdhsa_next_free_vgpr 136\n\t.end_amdhsa_kernel\n"
    assert asm_check.check(text, registers=[("kern", 136)]) == []
    assert asm_check.check(text, registers=[("kern", 128)]) == ["kernel: 136 registers, 128 at most"]
    assert asm_check.check(text, registers=[("other", 128)]) == ["no kernel is named like other"]
