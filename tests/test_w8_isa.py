"""The matrix-core and DPP distances of lrq_gemm_w8.hip's gfx950 build (CPU:
compiles to assembly), checked as the other kernel files' are."""

import os
import tempfile

import isa_hazards as H

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_w8_meets_wait_states():
    with tempfile.TemporaryDirectory() as d:
        text = H.compile_asm(os.path.join(ROOT, "loractl_amd", "csrc", "lrq_gemm_w8.hip"),
                             os.path.join(ROOT, "include"), d)
    total, bad = 0, []
    for k in H.parse_asm(text):
        v, n = H.check_kernel(k)
        total += n
        bad += v + H.check_dpp(k)[0]
    assert total > 0 and not bad, bad[:5]
