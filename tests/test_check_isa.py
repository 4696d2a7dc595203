"""The build's check of asm-issued matrix-core instructions (co-rope_amd/check_isa.py), on small pieces of assembly, and what the compiler noted
of the kernels in the built library."""
import importlib
import re

import pytest

check = importlib.import_module("co-rope_amd.check_isa").check_asm_mfma
check_tile_loops = importlib.import_module("co-rope_amd.check_isa").check_tile_loops

ASM = "\t;;#ASMSTART\n\tv_mfma_f32_32x32x16_bf16 v[16:31], v[32:35], v[48:51], v[0:15]\n\t;;#ASMEND\n"
ACCUMULATE = "\tv_mfma_f32_32x32x16_bf16 v[16:31], v[36:39], v[52:55], v[16:31]\n"


def test_in_place_accumulate_is_accepted():
    assert check("kern:\n" + ASM + "\tds_read_b128 v[36:39], v40\n" + ACCUMULATE + "\tv_mov_b32 v63, v17\n") == []


def test_register_copy_right_behind_it_is_reported():
    # what a build with accumulators in the other half of the register file produced: the copy reads the old contents
    problems = check("kern:\n" + ASM + "\ts_nop 0\n\tv_accvgpr_write_b32 a0, v16\n" + ACCUMULATE)
    assert len(problems) == 1 and "kern" in problems[0] and "v_accvgpr_write_b32" in problems[0]


def test_overwrite_and_other_accumulator_are_reported():
    assert check("kern:\n" + ASM + "\tds_read_b128 v[28:31], v40\n" + ACCUMULATE)
    assert check("kern:\n" + ASM + "\tv_mfma_f32_32x32x16_bf16 v[64:79], v[36:39], v[52:55], v[16:31]\n")


def test_untouched_for_long_enough_is_accepted():
    assert check("kern:\n" + ASM + "\ts_nop 11\n\tv_mov_b32 v63, v17\n") == []
    assert check("kern:\n" + ASM + "\ts_nop 5\n\tv_mov_b32 v63, v17\n")


def test_both_sides_of_a_branch_are_followed():
    tail = "\ts_cbranch_scc1 .LBB0_1\n\tv_mov_b32 v61, v62\n.LBB0_1:                 ; %bb.1\n"
    assert check("kern:\n" + ASM + tail + ACCUMULATE) == []
    assert check("kern:\n" + ASM + tail + "\tv_mov_b32 v63, v17\n")
    # only the path that is not taken reads the result too early
    assert check("kern:\n" + ASM + "\ts_cbranch_scc1 .LBB0_1\n\tv_mov_b32 v63, v17\n.LBB0_1:\n" + ACCUMULATE)


def test_result_in_the_accumulation_half_and_operand_there_are_understood():
    asm = "\t;;#ASMSTART\n\tv_mfma_f32_32x32x16_bf16 v[16:31], v[32:35], a[48:51], v[16:31]\n\t;;#ASMEND\n"
    assert check("kern:\n" + asm + "\ts_nop 11\n\tv_exp_f32_e32 v3, v17\n") == []
    assert check("kern:\n" + asm + "\tv_exp_f32_e32 v3, v17\n")
    asm_a = "\t;;#ASMSTART\n\tv_mfma_f32_32x32x16_bf16 a[0:15], v[32:35], v[48:51], a[0:15]\n\t;;#ASMEND\n"
    assert check("kern:\n" + asm_a + "\tv_accvgpr_read_b32 v3, a4\n")
    assert check("kern:\n" + asm_a + "\tv_mov_b32 v4, v5\n" * 12 + "\tv_accvgpr_read_b32 v3, a4\n") == []


def test_addend_overwritten_while_it_may_still_be_read_is_reported():
    # the result lands beside the addend v[0:15]: a vector write to the addend right behind the instruction is too early
    assert check("kern:\n" + ASM + "\tv_mov_b32_e32 v3, v40\n" + ACCUMULATE)
    assert check("kern:\n" + ASM + "\tv_mov_b32_e32 v40, v41\n" * 8 + "\tv_mov_b32_e32 v3, v40\n") == []
    # reading the addend is fine
    assert check("kern:\n" + ASM + "\tv_mov_b32_e32 v40, v3\n" + ACCUMULATE) == []


def test_operand_written_right_in_front_is_reported():
    assert check("kern:\n\tv_cvt_pk_bf16_f32 v48, v60, v61\n" + ASM + ACCUMULATE)
    assert check("kern:\n\tv_cvt_pk_bf16_f32 v48, v60, v61\n\ts_nop 1\n" + ASM + ACCUMULATE) == []
    assert check("kern:\n\tds_read_b128 v[32:35], v40\n\ts_waitcnt lgkmcnt(0)\n" + ASM + ACCUMULATE) == []


def test_sources_with_asm_matrix_instructions_are_found():
    build = importlib.import_module("co-rope_amd.build")
    checked = {s for s in build.SOURCES if build.isa_checked(s)}
    assert {"rope_attn_fwd_pipe.hip", "rope_attn_fwd_pipe_acc.hip", "rope_attn_bwd.hip"} <= checked
    assert "rope_rotate.hip" not in checked and "abi.hip" not in checked


ITEMS = """_ZN6corope23rope_attn_bwd_dq_kernelILi256ELi4ELi32ELb1ELb1ELb0EEEvNS_9BwdParamsE: ; @kernel
; %bb.0:
	s_load_dword s0, s[4:5], 0x0
.LBB0_1:                                ; =>This Loop Header: Depth=1
                                        ;     Child Loop BB0_2 Depth 2
	scratch_load_dword v1, off, off
.LBB0_2:                                ;   Parent Loop BB0_1 Depth=1
                                        ; =>  This Inner Loop Header: Depth=2
	{header}
	v_mfma_f32_32x32x16_bf16 a[16:31], v[36:39], v[52:55], a[16:31]
; %bb.3:                                ;   in Loop: Header=BB0_2 Depth=2
	{inner}
	s_cbranch_scc1 .LBB0_2
; %bb.4:                                ;   in Loop: Header=BB0_1 Depth=1
	scratch_store_dword off, v1, off
	s_cbranch_scc1 .LBB0_1
; %bb.5:
	s_endpgm
.Lfunc_end0:
"""


def test_scratch_in_a_tile_loop_is_reported():
    """What a kernel spills at a change of items passes; in its tile loop, in the loop's first block or another, it does not."""
    nop, spill = "s_nop 0", "scratch_store_dword off, v2, off offset:4"
    assert check_tile_loops(ITEMS.format(header=nop, inner=nop)) == []
    for where in (dict(header=spill, inner=nop), dict(header=nop, inner=spill)):
        problems = check_tile_loops(ITEMS.format(**where))
        assert len(problems) == 1 and "1 scratch" in problems[0] and "dq_kernel" in problems[0]
    # kernels that do not claim it are not held to it
    assert check_tile_loops(ITEMS.format(header=spill, inner=spill).replace("ELb1ELb1ELb0E", "ELb1ELb0ELb0E")) == []


def _kernels_of_the_library(path):
    """What the compiler noted of every kernel in a built library: the AMDGPU note (type 32) of each code object, a msgpack map."""
    msgpack = pytest.importorskip("msgpack")
    with open(path, "rb") as f:
        data = f.read()
    kernels = {}
    for m in re.finditer(rb"\x07\0\0\0(....)\x20\0\0\0AMDGPU\0\0", data, re.S):
        note = msgpack.unpackb(data[m.end():m.end() + int.from_bytes(m.group(1), "little")], strict_map_key=False)
        for k in note["amdhsa.kernels"]:
            kernels[k[".name"]] = k
    return kernels


def test_corope_forward_kernels_keep_their_registers():
    """None of the Co-RoPE forward's forms sends more than a handful of registers through scratch memory (with 84 and more, in the loop over
    rows, they took up to half as long again)."""
    lib = importlib.import_module("co-rope_amd._lib").LIB_PATH
    kernels = {n: k for n, k in _kernels_of_the_library(lib).items() if "corope_gqa_fwd_kernel" in n}
    assert any("corope_f16" in n for n in kernels) and any("corope_f16" not in n for n in kernels)
    spilled = {n: k[".vgpr_spill_count"] for n, k in kernels.items() if k[".vgpr_spill_count"] > 4}
    assert not spilled, spilled


@pytest.mark.parametrize("kernels,most", [
    (r"corope_f16\d+rope_attn_fwd_pipe_kernelILi64ELb[01]ELi[48]ELb[01]ELb1E", 0),       # fp16 probabilities, D = 64
    (r"corope_f16\d+rope_attn_fwd_pipe_kernelILi128ELb[01]ELi8ELb[01]ELb1E", 16),        # D = 128, eight waves, whole and cut
    (r"corope_f16\d+rope_attn_fwd_pipe_kernelILi128ELb[01]ELi4ELb0ELb1E", 32),           # four waves
    (r"rope_attn_bwd_dq_kernelILi256ELi4ELi32ELb[01]ELb1ELb0E", 40),                     # D = 256 on rotated operands: dQ, whole blocks
    (r"rope_attn_bwd_dkdv_kernelILi256ELi4ELi32ELb[01]ELb1ELb1ELb1ELb[01]E", 8),         # dK+dV, whole and cut
])
def test_streamed_kernels_keep_their_registers(kernels, most):
    """What these kernels spill lies at their changes of items (the build looks at the tile loops); more of it than when they were measured would
    show there, where nothing overlaps it."""
    notes = _kernels_of_the_library(importlib.import_module("co-rope_amd._lib").LIB_PATH)
    found = {n: k[".vgpr_spill_count"] for n, k in notes.items() if re.search(kernels, n)}
    assert len(found) >= 2 and max(found.values()) <= most, found
