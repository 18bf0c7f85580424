"""The matrix-core and DPP distances of lrq_gemm_w8.hip's gfx950 build (CPU:
compiles to assembly), checked as the other kernel files' are, and
the wait for the copies before each barrier of its pipelined loop."""

import os
import re
import tempfile

import isa_hazards as H

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_w8_meets_wait_states():
    with tempfile.TemporaryDirectory() as d:
        text = H.compile_asm(os.path.join(ROOT, "loractl_amd", "csrc", "lrq_gemm_w8.hip"),
                             os.path.join(ROOT, "include"), d)
    total, bad = 0, []
    for k in H.parse_asm(text):
        # a stage's barrier publishes the next stage's LDS copies: they have landed
        waits = H.stage_waits(k)
        assert "k_w8" not in k.name or (waits and all(w == 0 for w, _ in waits)), (k.name, waits)
        v, n = H.check_kernel(k)
        total += n
        bad += v + H.check_dpp(k)[0]
    assert total > 0 and not bad, bad[:5]
    # the side products' registers stay within the tiles': no spills to scratch
    spills = re.findall(r"^\s*\.vgpr_spill_count:\s*(\d+)", text, flags=re.M)
    assert spills and not any(int(s) for s in spills), spills
