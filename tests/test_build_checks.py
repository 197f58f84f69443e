"""The build's checks of compiler output, on short listings (no compiler needed)."""
import importlib.util
import os

import pytest

_spec = importlib.util.spec_from_file_location("_build_checks", os.path.join(os.path.dirname(__file__), "..", "llm-systems-from-scratch_amd", "build.py"))
build = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(build)

MFMA = "v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]"
CONVERT = "v_cvt_pk_bf16_f32 v8, v9, v10"


def _asm(*text):
    return ["\t;;#ASMSTART", *("\t" + t for t in text), "\t;;#ASMEND"]


@pytest.mark.parametrize("lines,right", [
    ([*_asm(MFMA)], True), (["\tv_mov_b32_e32 v4, 0", *_asm(MFMA)], False), (["\tv_mov_b32_e32 v4, 0", "\ts_nop 1", *_asm(MFMA)], True), (["\tv_mov_b32_e32 v8, 0", *_asm(MFMA)], True),
    ([*_asm("v_cvt_pk_bf16_f32 v7, v9, v10"), *_asm(MFMA)], False), ([*_asm(MFMA), *_asm(MFMA)], True), ([*_asm(MFMA), "\tv_accvgpr_read_b32 v9, a3"], False),
    ([*_asm(MFMA), "\ts_nop 15", "\tv_accvgpr_read_b32 v9, a3"], True), (["\tv_exp_f32_e32 v9, v9", *_asm(CONVERT)], False),
    (["\tv_exp_f32_e32 v9, v9", "\tv_mul_f32_e32 v1, v2, v3", *_asm(CONVERT)], True), (["\tv_mul_f32_e32 v9, v9, v3", *_asm(CONVERT)], True),
    (["\tv_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], 0", *_asm(CONVERT)], False), (["\tv_mfma_f32_32x32x16_bf16 v[16:31], v[20:23], v[24:27], 0", *_asm(CONVERT)], True)])
def test_hazards_of_inline_assembly(lines, right):
    n_mfma, n_other, bad = build.asm_hazards(lines)
    assert n_mfma + n_other >= 1 and bool(bad) != right, bad


def test_without_markers_nothing_is_found():
    """(the build fails then: it expects a number of them)"""
    assert build.asm_hazards(["\tv_mov_b32_e32 v4, 0", "\t" + MFMA]) == (0, 0, [])


SPILL = "\tscratch_store_dword off, v1, off offset:4 ; 4-byte Folded Spill"


@pytest.mark.parametrize("where,right", [("front", False), ("loop", False), ("aside", False), ("behind", True)])
def test_spills_before_the_last_product(where, right):
    lines = ["_Z5otherv:", SPILL, "\t" + MFMA, "\ts_endpgm", ".Lfunc_end0:", "_Z6kernelv:                             ; @_Z6kernelv", *([SPILL] * (where == "front")), ".LBB1_1:",
             "\ts_cbranch_scc1 .LBB1_3", ".LBB1_2:", "\t" + MFMA, *([SPILL] * (where == "loop")), "\ts_cbranch_vccnz .LBB1_1", *([SPILL] * (where == "behind")), "\ts_endpgm", ".LBB1_3:",
             *([SPILL] * (where == "aside")), "\ts_branch .LBB1_2", ".Lfunc_end1:", "_Z4lastv:", SPILL, "\t" + MFMA]
    assert bool(build.scratch_before_products(lines, "kernel")) != right
    assert build.scratch_before_products(lines, "missing") is None
