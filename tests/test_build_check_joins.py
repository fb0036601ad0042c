"""The build's check of the compiler's output at the joins that do not end an if: the end of a
loop, where no lane is left, and an else."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "hyqmom.jl_amd"))
from build import masked_copies  # noqa: E402

# {0}: before the mask is restored; {1}: after
LOOP = """k:                                      ; @k
.LBB0_1:
\tv_add_u32_e32 v1, -1, v1
\tv_cmp_eq_u32_e32 vcc, 0, v1
\ts_or_b64 s[2:3], vcc, s[2:3]
\ts_andn2_b64 exec, exec, s[2:3]
\ts_cbranch_execnz .LBB0_1
; %bb.2:
{0}\ts_or_b64 exec, exec, s[2:3]
{1}\ts_endpgm
.Lfunc_end0:
"""
# a loop over the distinct values of a register
VALUES = LOOP.replace("s_andn2_b64 exec, exec, s[2:3]", "s_xor_b64 exec, exec, s[2:3]").replace(
    "s_or_b64 exec, exec, s[2:3]\n{1}", "s_mov_b64 exec, s[2:3]\n{1}")
# the loop's exit reached from elsewhere too
LABEL = LOOP.replace("; %bb.2:", ".LBB0_2:")
ELSE = """k:                                      ; @k
\ts_and_saveexec_b64 s[2:3], vcc
\ts_xor_b64 s[2:3], exec, s[2:3]
\ts_cbranch_execz .LBB0_2
; %bb.1:
\tv_add_f64 v[4:5], v[4:5], v[6:7]
.LBB0_2:
{0}\ts_or_saveexec_b64 s[2:3], s[2:3]
{1}\ts_xor_b64 exec, exec, s[2:3]
\ts_endpgm
.Lfunc_end0:
"""
COPY = "\tv_accvgpr_write_b32 a28, v70\n"


@pytest.mark.parametrize("asm", [LOOP, VALUES, LABEL, ELSE], ids=["loop", "values", "label", "else"])
@pytest.mark.parametrize("copy", [COPY, "\tscratch_store_dword off, v70, off offset:4\n"])
def test_copies_at_loop_ends_and_elses(asm, copy):
    assert masked_copies(asm.format("", copy)) == []
    assert [(f, v) for f, _, v in masked_copies(asm.format("\ts_mov_b32 s18, 0\n" + copy, ""))] == [("k", [copy.strip()])]


def test_values_of_the_then_side_may_move_before_an_else():
    move = "\tv_mov_b32_e32 v9, v4\n"
    assert masked_copies(ELSE.format(move, "")) == []
    assert masked_copies(LOOP.format(move, "")) != []  # no lane is left to move it


def test_a_branch_that_is_always_taken_ends_no_loop():
    asm = LOOP.replace("\ts_andn2_b64 exec, exec, s[2:3]\n", "\ts_mov_b64 vcc, exec\n")
    assert masked_copies(asm.format(COPY, "")) == []
