"""The build-time assembly check must catch a register that is touched while an inline-assembly
load into it is still in flight, and must accept the same code once a counted wait covers it."""
import pytest

from lmdeploy_amd.asm_lint import lint

HEAD = "_ZN5w4a164test_kernelEv:\n"
TAIL = "\ts_endpgm\n.Lfunc_end0:\n"


def load(reg):
    return "\t;;#ASMSTART\n\tglobal_load_dwordx4 v[%d:%d], v40, s[2:3] offset:0\n\t;;#ASMEND\n" % (reg, reg + 3)


def test_clean_counted_wait():
    asm = HEAD + load(0) + load(4) + "\ts_waitcnt vmcnt(1)\n\tv_mov_b32_e32 v20, v1\n" + TAIL
    assert lint(asm) == []


def test_copy_before_wait_is_reported():
    asm = HEAD + load(0) + load(4) + "\tv_mov_b32_e32 v20, v1\n\ts_waitcnt vmcnt(1)\n" + TAIL
    msgs = lint(asm)
    assert len(msgs) == 1 and "v1" in msgs[0]


def test_wait_too_weak_is_reported():
    # vmcnt(1) retires only the older load: v[4:7] may still be in flight
    asm = HEAD + load(0) + load(4) + "\ts_waitcnt vmcnt(1)\n\tv_add_u32_e32 v21, v5, v5\n" + TAIL
    assert len(lint(asm)) == 1


def test_loop_carried_load_is_tracked_across_the_back_edge():
    # the load at the end of the loop body is in flight at the top of the next trip
    asm = (HEAD + load(0) + ".LBB0_1:\n\ts_waitcnt vmcnt(0)\n\tv_mov_b32_e32 v20, v0\n" + load(0)
           + "\tv_mov_b32_e32 v21, v2\n\ts_cbranch_scc1 .LBB0_1\n" + TAIL)
    msgs = lint(asm)
    assert len(msgs) == 1 and "v_mov_b32_e32 v21, v2" in msgs[0]


def test_join_takes_the_younger_position():
    # one path issues a second load, so after the join vmcnt(1) no longer covers v[0:3]... it does:
    # v[0:3] is older on both paths; v[4:7] is only in flight on one of them and must stay flagged
    asm = (HEAD + load(0) + "\ts_cbranch_scc1 .LBB0_2\n" + load(4) + ".LBB0_2:\n\ts_waitcnt vmcnt(1)\n"
           "\tv_mov_b32_e32 v20, v4\n" + TAIL)
    assert len(lint(asm)) == 1


def test_other_functions_are_ignored():
    asm = "_ZN5w4a166helperEv:\n" + load(0) + "\tv_mov_b32_e32 v20, v1\n" + TAIL
    assert lint(asm) == []


def test_parking_an_in_flight_register_in_an_agpr_is_reported():
    # the register allocator saves a VGPR to an AGPR to reuse it, while a load into it is pending:
    # the saved value is stale and the load later lands on the register's new owner
    asm = HEAD + load(48) + "\tv_accvgpr_write_b32 a106, v51\n\ts_waitcnt vmcnt(0)\n" + TAIL
    msgs = lint(asm)
    assert len(msgs) == 1 and "v51" in msgs[0]


def test_parking_a_settled_register_is_accepted():
    asm = HEAD + load(48) + "\ts_waitcnt vmcnt(0)\n\tv_accvgpr_write_b32 a106, v51\n" + TAIL
    assert lint(asm) == []


def mfma(acc):
    return "\t;;#ASMSTART\n\tv_mfma_f32_16x16x32_f16 a[%d:%d], v[0:3], v[4:7], a[%d:%d]\n\t;;#ASMEND\n" % (acc, acc + 3, acc, acc + 3)


def test_accumulator_read_right_after_an_inline_mfma_is_reported():
    asm = HEAD + mfma(8) + "\tv_accvgpr_read_b32 v20, a9\n" + TAIL
    msgs = lint(asm)
    assert len(msgs) == 1 and "wait states" in msgs[0]


def test_accumulator_read_after_the_pipe_has_drained_is_accepted():
    asm = HEAD + mfma(8) + "\t;;#ASMSTART\n\ts_nop 15\n\ts_nop 15\n\t;;#ASMEND\n\tv_accvgpr_read_b32 v20, a9\n" + TAIL
    assert lint(asm) == []


def test_accumulator_move_inside_a_loop_of_inline_mfmas_is_reported():
    # at the top of the body, textually before the MFMA, but reached again across the back edge
    asm = (HEAD + ".LBB0_1:\n\tv_accvgpr_mov_b32 a8, a12\n" + mfma(8) + "\ts_cbranch_scc1 .LBB0_1\n" + TAIL)
    msgs = lint(asm)
    assert any("inside a loop" in m for m in msgs)


def test_a_register_range_is_seen():
    asm = HEAD + load(12) + "\tv_mov_b64_e32 v[40:41], v[14:15]\n\ts_waitcnt vmcnt(0)\n" + TAIL
    assert len(lint(asm)) == 1


def test_lds_reads_are_waited_for_by_count():
    read = "\t;;#ASMSTART\n\tds_read_b128 v[%d:%d], v40 offset:0\n\t;;#ASMEND\n"
    asm = HEAD + read % (0, 3) + read % (4, 7) + "\ts_waitcnt lgkmcnt(1)\n\tv_mov_b32_e32 v20, v1\n" + TAIL
    assert lint(asm) == []
    asm = HEAD + read % (0, 3) + read % (4, 7) + "\ts_waitcnt lgkmcnt(1)\n\tv_mov_b32_e32 v20, v5\n" + TAIL
    assert len(lint(asm)) == 1


def test_m0_written_by_the_compiler_where_loads_rely_on_it_is_reported():
    put = "\t;;#ASMSTART\n\ts_mov_b32 m0, s5\n\ts_nop 0\n\t;;#ASMEND\n"
    dma = "\t;;#ASMSTART\n\tglobal_load_lds_dwordx4 v40, s[2:3] offset:1024\n\t;;#ASMEND\n"
    both = "\t;;#ASMSTART\n\ts_mov_b32 m0, s5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 v40, s[2:3]\n\t;;#ASMEND\n"
    other = "\ts_mov_b32 m0, s9\n"
    assert lint(HEAD + put + dma + dma + TAIL) == []
    assert lint(HEAD + both + other + both + TAIL) == []                # (every statement sets its own)
    assert lint(HEAD + put + dma + "\ts_cmp_eq_u32 m0, s9\n" + dma + TAIL) == []
    msgs = lint(HEAD + put + dma + other + dma + TAIL)
    assert len(msgs) == 1 and "writes M0" in msgs[0]


def test_lds_exchanges_need_a_barrier():
    put, get = "\tds_write_b128 v2, v[4:7]\n", "\tds_read_b128 v[8:11], v3\n"
    for between in ("\t; wave barrier\n", "\ts_barrier\n"):
        assert lint(HEAD + get + put + between + get + TAIL) == []
        # (a barrier on one of two ways is none)
        assert len(lint(HEAD + put + "\ts_cbranch_scc1 .LBB0_1\n" + between + ".LBB0_1:\n" + get + TAIL)) == 1
    msgs = lint(HEAD + put + get + TAIL)
    assert len(msgs) == 1 and "no barrier between" in msgs[0]
    # across the back edge of a loop
    assert len(lint(HEAD + ".LBB0_1:\n" + get + put + "\ts_cbranch_scc1 .LBB0_1\n" + TAIL)) == 1
    assert lint(HEAD + ".LBB0_1:\n\t; wave barrier\n" + get + put + "\ts_cbranch_scc1 .LBB0_1\n" + TAIL) == []


def test_the_conversion_is_checked():
    from lmdeploy_amd import build
    assert "repack.hip" in build.LINTED


MASKED = "\t;;#ASMSTART\n\ts_mov_b64 exec, s[40:41]\n\tglobal_load_dword v0, v40, s[2:3]\n\ts_mov_b64 exec, -1\n\t;;#ASMEND\n"
BRANCH = "\ts_and_saveexec_b64 s[10:11], vcc\n\ts_cbranch_execz .LBB0_1\n%s.LBB0_1:\n\ts_or_b64 exec, exec, s[10:11]\n"
BOTH = ("\ts_and_saveexec_b64 s[10:11], vcc\n\ts_xor_b64 s[10:11], exec, s[10:11]\n\tv_mov_b32_e32 v30, 0\n"
        "\ts_andn2_saveexec_b64 s[10:11], s[10:11]\n\ts_cbranch_execz .LBB0_1\n%s.LBB0_1:\n\ts_or_b64 exec, exec, s[10:11]\n")
LOOP = ("\ts_mov_b64 s[20:21], 0\n.LBB0_7:\n%s\tv_cmp_gt_u32_e32 vcc, v30, v31\n\ts_or_b64 s[20:21], vcc, s[20:21]\n"
        "\ts_andn2_b64 exec, exec, s[20:21]\n\ts_cbranch_execnz .LBB0_7\n\ts_or_b64 exec, exec, s[20:21]\n")
INNER = "\ts_and_saveexec_b64 s[12:13], s[14:15]\n\tv_mov_b32_e32 v30, 0\n\ts_or_b64 exec, exec, s[12:13]\n"


@pytest.mark.parametrize("body", [MASKED, MASKED + MASKED, BRANCH % "" + MASKED, BRANCH % INNER + MASKED, BOTH % INNER + MASKED, BRANCH % LOOP % "" + MASKED,
                                  "\ts_mov_b64 s[6:7], exec\n\ts_and_b64 exec, exec, vcc\n\ts_mov_b64 exec, s[6:7]\n" + MASKED,
                                  ".LBB0_2:\n" + BRANCH % INNER + MASKED + "\ts_cbranch_scc1 .LBB0_2\n"])
def test_masked_loads_where_every_lane_is_active(body):
    assert lint(HEAD + body + TAIL) == []


@pytest.mark.parametrize("body", [
    BRANCH % MASKED, BOTH % MASKED, BRANCH % (INNER + MASKED), BRANCH % LOOP % MASKED,
    "\ts_and_b64 exec, exec, vcc\n" + MASKED,
    "\ts_mov_b64 exec, s[6:7]\n" + MASKED,
    "\ts_mov_b32 exec_lo, s6\n" + MASKED,
    BRANCH % "\ts_mov_b32 s11, 0\n" + MASKED,                                  # the saved mask was written over
    BRANCH % "\tv_add_co_u32_e64 v30, s[10:11], v30, v31\n" + MASKED,
    "\ts_and_saveexec_b64 s[10:11], vcc\n\ts_cbranch_scc1 .LBB0_1\n\ts_or_b64 exec, exec, s[10:11]\n.LBB0_1:\n" + MASKED,   # restored on one way
    ".LBB0_2:\n" + MASKED + "\ts_and_b64 exec, exec, vcc\n\ts_cbranch_execnz .LBB0_2\n",                                   # around the back edge
    LOOP % ("\ts_and_saveexec_b64 s[12:13], vcc\n\ts_xor_b64 s[16:17], exec, s[12:13]\n") + "\ts_or_b64 exec, exec, s[16:17]\n" + MASKED])
def test_masked_loads_where_a_lane_may_be_off_are_reported(body):
    msgs = lint(HEAD + body + TAIL)
    assert len(msgs) == 1 and "switches every lane on" in msgs[0]
