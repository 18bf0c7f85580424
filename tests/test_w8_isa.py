"""The matrix-core and DPP distances of lrq_gemm_w8.hip's gfx950 build (CPU:
compiles to assembly), checked as the other kernel files' are, and
the wait for the copies before each barrier of its pipelined loop."""

import os
import re
import tempfile

import isa_hazards as H

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copy_checker_follows_paths():
    """A copy past a wait that a branch skips, and one behind the wait."""
    copy = "\tbuffer_load_dwordx4 v1, s[0:3], 0 offen lds\n"
    listing = ("\t.text\n\t.globl k\n\t.type k,@function\nk:\n" + copy + "\ts_cbranch_scc1 .LBB0_2\n"
               "\ts_waitcnt vmcnt(0)\n{}.LBB0_2:\n\ts_barrier\n\ts_endpgm\n.Lfunc_end0:\n")
    assert [j for _, j in H.unwaited_copies(H.parse_asm(listing.format(""))[0])] == [3]
    assert [i for i, _ in H.unwaited_copies(H.parse_asm(listing.format(copy))[0])] == [0, 3]
    waited = listing.format("").replace("\ts_cbranch_scc1", "\ts_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_cbranch_scc1")
    assert not H.unwaited_copies(H.parse_asm(waited)[0])


def test_w8_meets_wait_states():
    with tempfile.TemporaryDirectory() as d:
        text = H.compile_asm(os.path.join(ROOT, "loractl_amd", "csrc", "lrq_gemm_w8.hip"),
                             os.path.join(ROOT, "include"), d)
    total, bad = 0, []
    for k in H.parse_asm(text):
        # a stage's barrier publishes the next stage's LDS copies: they have landed
        waits = H.stage_waits(k)
        assert "k_w8" not in k.name or (waits and all(w == 0 for w, _ in waits)), (k.name, waits)
        # and so does every copy's, on every path (the tail stage's, whose LDS
        # the depth groups' sums reuse)
        assert not H.unwaited_copies(k), (k.name, H.unwaited_copies(k)[:3])
        v, n = H.check_kernel(k)
        total += n
        bad += v + H.check_dpp(k)[0]
    assert total > 0 and not bad, bad[:5]
    # the side products' registers stay within the tiles': no spills to scratch
    spills = re.findall(r"^\s*\.vgpr_spill_count:\s*(\d+)", text, flags=re.M)
    assert spills and not any(int(s) for s in spills), spills
