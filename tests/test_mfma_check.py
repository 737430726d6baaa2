"""The build-time scans for early readers of matrix products and of other lanes' registers (int_flashattention_amd/mfma_check.py) on hand-made assembly: a product of four
passes (16 x 16) needs eight wait states, one of eight passes (32 x 32) twelve, on every way to an instruction that touches its registers."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "int-flashattention_amd"))
import mfma_check  # noqa: E402

HEAD = "_ZN5intfa4kernEv:\n\ts_load_dwordx2 s[0:1], s[4:5], 0x0\n"
SMALL = "\tv_mfma_f32_16x16x32_f16 v[0:3], v[8:11], v[12:15], v[0:3]\n"
LARGE = "\tv_mfma_i32_32x32x32_i8 v[16:31], v[8:11], v[12:15], 0\n"


@pytest.mark.parametrize("product,states,reader", [
    (SMALL, 8, "v_mul_f32_e32 v4, v3, v5"), (SMALL, 8, "ds_write_b128 v7, v[0:3]"), (SMALL, 8, "v_mov_b32_e32 v0, 0"),
    (SMALL, 8, "v_mfma_f32_16x16x32_f16 v[32:35], v[0:3], v[12:15], 0"), (SMALL, 8, "v_mfma_f32_16x16x32_f16 v[32:35], v[8:11], v[12:15], v[2:5]"),
    (LARGE, 12, "v_cvt_f32_i32_e32 v4, v16"), (LARGE, 12, "global_store_dword v[4:5], v31, off"), (LARGE, 12, "v_accvgpr_write_b32 a0, v20"),
])
def test_the_last_wait_state_counts(product, states, reader):
    for have in (0, states - 1, states):
        nops = "".join("\ts_mov_b32 s9, s8\n" for _ in range(have % 4)) + (f"\ts_nop {have - have % 4 - 1}\n" if have >= 4 else "")
        found = mfma_check.scan(HEAD + product + nops + "\t" + reader + " ; a comment naming v0\n\ts_endpgm\n")
        assert len(found) == (have < states), (have, found)
        assert all(f"{states - have} wait states too early" in f and "_ZN5intfa4kernEv" in f for f in found)


def test_a_chain_and_other_registers_need_no_wait():
    asm = (HEAD + LARGE + "\tv_mfma_i32_32x32x32_i8 v[16:31], v[8:11], v[12:15], v[16:31]\n"
           "\tv_mfma_i32_32x32x32_i8 v[40:55], v[8:11], v[12:15], v[16:31]\n\tv_add_f32_e32 v1, v2, v15\n\tv_mov_b32_e32 v32, s16\n\ts_endpgm\n")
    assert mfma_check.scan(asm) == []
    # accumulation registers are registers of their own
    acc = HEAD + LARGE.replace("v[16:31]", "a[16:31]") + "\tv_mov_b32_e32 v16, 0\n\t{}\n\ts_endpgm\n"
    assert mfma_check.scan(acc.format("s_nop 0")) == []
    assert len(mfma_check.scan(acc.format("v_accvgpr_read_b32 v0, a16"))) == 1


# A product, a way around other products, the reader: the wait must be there on the short way too.
SKIP = ("\ts_cbranch_scc1 .LBB0_2\n; %bb.1:\n" + 12 * "\tv_mov_b32_e32 v60, 0\n" + ".LBB0_2:\n")


def test_the_shorter_of_two_ways_counts():
    reader = "\tv_cvt_f32_i32_e32 v4, v16\n\ts_endpgm\n"
    assert len(mfma_check.scan(HEAD + LARGE + SKIP + reader)) == 1
    assert len(mfma_check.scan(HEAD + LARGE + SKIP + "\ts_nop 9\n" + reader)) == 1
    assert mfma_check.scan(HEAD + LARGE + SKIP + "\ts_nop 10\n" + reader) == []


def test_a_loop_and_its_exit_are_followed():
    loop = HEAD + ".LBB0_1:\n\tv_mul_f32_e32 v1, v1, v5\n" + 8 * "\ts_mov_b32 s9, s8\n" + SMALL + "{}\ts_cbranch_scc1 .LBB0_1\n; %bb.2:\n{}\tv_add_f32_e32 v6, v0, v0\n\ts_endpgm\n"
    found = mfma_check.scan(loop.format("", "\ts_nop 6\n"))
    assert len(found) == 1 and "v_mul_f32_e32 v1" in found[0]      # the next round reads too early, the code behind the loop does not
    found = mfma_check.scan(loop.format("\ts_nop 6\n", ""))
    assert found == []
    found = mfma_check.scan(loop.format("\ts_nop 5\n", ""))
    assert len(found) == 2


def test_an_unknown_product_is_reported():
    found = mfma_check.scan(HEAD + "\tv_mfma_f64_16x16x4_f64 v[0:7], v[8:9], v[10:11], v[0:7]\n\ts_endpgm\n")
    assert len(found) == 1 and "table" in found[0]


def test_a_wait_for_loads_ahead_of_a_product_in_a_loop_is_reported():
    """Q is fetched ahead of the loop; the compiler's wait for it belongs there too."""
    head = HEAD + "\tglobal_load_dwordx4 v[12:15], v[60:61], off\n{}.LBB0_1: ; =>This Inner Loop Header: Depth=1\n"
    copy = "\t;;#ASMSTART\n\ts_waitcnt vmcnt(0)\n\t;;#ASMEND\n\ts_barrier\n\t;;#ASMSTART\n\tbuffer_load_dwordx4 v70, s[8:11], s12 offen lds\n\t;;#ASMEND\n"
    end = LARGE + "\ts_cbranch_scc1 .LBB0_1\n; %bb.2:\n\ts_endpgm\n"
    found = mfma_check.scan_waits(head.format("") + copy + "\ts_waitcnt vmcnt(0) lgkmcnt(1)\n" + end)
    assert len(found) == 1 and "_ZN5intfa4kernEv" in found[0]
    assert mfma_check.scan_waits(head.format("\ts_waitcnt vmcnt(0)\n") + copy + "\ts_waitcnt lgkmcnt(1)\n" + end) == []
    assert mfma_check.scan_waits(HEAD + "\ts_waitcnt vmcnt(0)\n" + LARGE + "\ts_endpgm\n") == []      # not in a loop
    spilled = "\tscratch_load_dwordx4 v[12:15], off, off offset:16 ; 16-byte Folded Reload\n\ts_waitcnt vmcnt(0)\n"
    assert mfma_check.scan_waits(head.format("") + copy + spilled + end) == []


LANES = "\tv_fmac_f32_dpp v7, v1, v9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"


@pytest.mark.parametrize("writer,states", [("v_mov_b32_e32 v1, v50", 2), ("v_accvgpr_read_b32 v1, a3", 2), ("v_cmpx_gt_f32_e32 v2, v3", 5)])
def test_another_lanes_register_is_not_read_too_early(writer, states):
    for have in range(states + 1):
        nops = f"\ts_nop {have - 1}\n" if have else ""
        found = mfma_check.scan_lanes(HEAD + f"\t{writer}\n" + nops + LANES + "\ts_endpgm\n")
        assert len(found) == (have < states), (have, found)
        assert all(f"{states - have} wait states too early" in f and "_ZN5intfa4kernEv" in f for f in found)


def test_only_the_lanes_source_waits():
    # loads from the LDS are waited for; the other source and the addend are the lane's own; instructions without DPP read what they like
    for writer in ("ds_read_b32 v1, v2", "v_mov_b32_e32 v9, 0", "v_mov_b32_e32 v7, 0", "v_cmp_gt_f32_e32 vcc, v1, v3", "s_mov_b32 s1, s2"):
        assert mfma_check.scan_lanes(HEAD + f"\t{writer}\n" + LANES + "\ts_endpgm\n") == []
    assert mfma_check.scan_lanes(HEAD + "\tv_mov_b32_e32 v1, v50\n\tv_add_f32_e32 v3, v1, v1\n" + "\ts_nop 0\n" + LANES + "\ts_endpgm\n") == []
    # (operands of several registers, and the modifier in the place of the suffix)
    wide = HEAD + "\tv_lshlrev_b64 v[0:1], 1, v[4:5]\n\tv_mov_b32 v7, v1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\ts_endpgm\n"
    assert len(mfma_check.scan_lanes(wide)) == 1


def test_another_lanes_register_on_every_way():
    asm = HEAD + "\tv_mov_b32_e32 v1, v50\n{}" + SKIP + "{}" + LANES + "\ts_endpgm\n"
    # (the branch is a wait state)
    assert len(mfma_check.scan_lanes(asm.format("", ""))) == 1
    assert mfma_check.scan_lanes(asm.format("\ts_nop 0\n", "")) == []
    assert mfma_check.scan_lanes(asm.format("", "\ts_nop 0\n")) == []
    # over the back edge of a loop
    loop = HEAD + ".LBB0_1:\n" + LANES + 4 * "\ts_mov_b32 s9, s8\n" + "\tv_mov_b32_e32 v1, v50\n{}\ts_cbranch_scc1 .LBB0_1\n; %bb.2:\n\ts_endpgm\n"
    assert len(mfma_check.scan_lanes(loop.format(""))) == 1
    assert mfma_check.scan_lanes(loop.format("\ts_nop 0\n")) == []
