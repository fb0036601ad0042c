"""The build's check of the compiler's output: vector copies in a join block, ahead of the
restored execution mask."""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "hyqmom.jl_amd"))
from build import masked_copies  # noqa: E402

GOOD = """k:                                      ; @k
\tv_cmp_ne_u32_e32 vcc, 0, v1
\ts_and_saveexec_b64 s[2:3], vcc
\ts_cbranch_execz .LBB0_2
; %bb.1:
\tv_mov_b32_e32 v0, v2
.LBB0_2:
\ts_or_b64 exec, exec, s[2:3]
\tv_accvgpr_write_b32 a28, v70
.Lfunc_end0:
"""


def test_copies_after_the_mask_are_fine():
    assert masked_copies(GOOD) == []


def test_copies_before_the_mask_are_found():
    bad = GOOD.replace("\ts_or_b64 exec, exec, s[2:3]\n\tv_accvgpr_write_b32 a28, v70\n",
                       "\tv_accvgpr_write_b32 a28, v70\n\ts_mov_b32 s18, 0\n\ts_or_b64 exec, exec, s[2:3]\n")
    assert [(f, v) for f, _, v in masked_copies(bad)] == [("k", ["v_accvgpr_write_b32 a28, v70"])]
    # the same without a branch over the narrowed block
    fall = bad.replace("\ts_cbranch_execz .LBB0_2\n", "").replace(".LBB0_2:", "; %bb.2:")
    assert [(f, v) for f, _, v in masked_copies(fall)] == [("k", ["v_accvgpr_write_b32 a28, v70"])]
