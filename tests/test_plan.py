"""How calls plan their kernel and workspace, through the host-only planner
hook (no GPU)."""

import itertools
import random

import pytest

from loractl_amd import _lib as L
from loractl_amd import device as D

SCRATCH = L.LRQ_NOALLOC_SCRATCH_BYTES - (64 << 10)  # past the arrival counters
TOKENS = [17, 96, 192, 320, 512, 640, 896, 1024, 1792, 2112, 4096, 8192]
FORMATS = (L.LRQ_FMT_INT4, L.LRQ_FMT_INT8, L.LRQ_FMT_FP8)
DIMS = [512, 2560, 3072, 4096, 9216, 12288, 14336, 16384, 18432]


@pytest.mark.parametrize("m,k,n,r", [(64, 18432, 12288, 64), (640, 18432, 2560, 64), (1024, 14336, 2560, 32),
                                     (8192, 12288, 2560, 32), (8192, 12288, 9216, 32)])
def test_noalloc_plans_a_kernel_that_fits(m, k, n, r):
    """The fastest plan of these needs more than the scratch; another fits."""
    assert D.debug_plan("fwd", m, n, k, r)["bytes"] > SCRATCH
    assert D.debug_plan("noalloc", m, n, k, r)["bytes"] <= SCRATCH


def test_noalloc_takes_the_ordinary_plan_where_it_fits():
    for m, k, n, r in itertools.product(TOKENS, DIMS, DIMS, (16, 32, 64)):
        p, q = D.debug_plan("fwd", m, n, k, r), D.debug_plan("noalloc", m, n, k, r)
        keys = ("bytes", "kernel", "ranges", "folded")
        if p["bytes"] <= SCRATCH:
            assert all(p[x] == q[x] for x in keys), (m, k, n, r)
        assert q["bytes"] <= SCRATCH, (m, k, n, r)


@pytest.mark.parametrize("what,m,n,k", [("bwd", 100000, 21512, 512), ("bwd", 100000, 18440, 512), ("bwd", 80000, 18440, 128),
                                        ("fwd", 100000, 512, 18432)])
def test_folded_factors_stay_within_32_bit_offsets(what, m, n, k):
    """Activations of 2 GiB and more (the folded factor's masked loads use
    that offset) take side launches; smaller ones fold."""
    for r in (8, 16, 32):
        assert not D.debug_plan(what, m, n, k, r)["folded"]
        assert D.debug_plan(what, 2048, 1536, 1536, r)["folded"]


@pytest.mark.parametrize("n,k", [(12288, 3072), (3072, 12288), (3072, 3072), (9728, 2560), (8192, 512), (520, 96)])
def test_reserve_covers_every_smaller_token_count(n, k):
    """Also at counts inside a 64-token group, past the kernels' tiles."""
    rng = random.Random(n + k)
    for r in (0, 8, 16, 17, 32, 64):
        for m in (1, 16, 100, 512, 1000, 1024, 2048, 4096):
            have = D.debug_plan("reserve", m, n, k, r)["bytes"]
            counts = set(range(64, m, 64)) | {m} | {rng.randint(1, m) for _ in range(200)}
            for q in counts:
                need = max(D.debug_plan(w, q, n, k, r, f)["bytes"] for w in ("fwd", "bwd") for f in FORMATS)
                assert need <= have, (m, q, r, need, have)


def test_depth_ranges_have_a_place_each():
    """Ranges only where all their workgroups run at once (256 CUs, two of the
    64-row tiles' workgroups on each): at most 256 tiles of 256 x 128 partials."""
    rows, tokens, places = {1: 64, 2: 128, 3: 256, 4: 64}, {1: 64, 2: 128, 3: 128, 4: 128}, {1: 512, 2: 256, 3: 256, 4: 512}
    seen = set()
    for m, k, n, r in itertools.product(TOKENS, DIMS, DIMS, (0, 16, 32)):
        for what, e in (("fwd", n), ("bwd", k)):
            p = D.debug_plan(what, m, n, k, r)
            v = p["kernel"]
            seen.add((v, p["ranges"] > 1))
            if v and p["ranges"] > 1:
                units = -(-m // tokens[v]) * -(-e // rows[v]) * p["ranges"]
                assert units <= places[v], (what, m, k, n, r, p)
            if v and r == 0:
                assert p["bytes"] <= 256 * 256 * 128 * 4
    assert {(1, True), (2, True), (3, True), (4, True), (0, True), (3, False)} <= seen


# calls that a model without the factors' workgroups, or without the format,
# sent to kernels 1.2 to 1.7 times as slow as the fastest; the plans measured
# within a tenth of it
MEASURED = [
    ("bwd", 128, 12288, 3072, 32, L.LRQ_FMT_INT4, {(1, 4), (2, 6)}),
    ("bwd", 256, 12288, 3072, 32, L.LRQ_FMT_INT4, {(2, 3), (2, 4), (4, 4)}),
    ("bwd", 512, 4096, 2560, 0, L.LRQ_FMT_INT4, {(2, 2), (2, 3)}),
    ("bwd", 384, 512, 8192, 16, L.LRQ_FMT_INT4, {(4, 1)}),
    ("fwd", 384, 3072, 3072, 16, L.LRQ_FMT_INT4, {(2, 2), (2, 3)}),
    ("bwd", 3868, 10744, 576, 24, L.LRQ_FMT_INT4, {(0, 1), (2, 1), (3, 2)}),
    ("bwd", 3301, 13712, 672, 32, L.LRQ_FMT_FP8, {(0, 1), (2, 1), (3, 2), (3, 3)}),
    ("fwd", 59, 1144, 11968, 32, L.LRQ_FMT_FP8, {(1, 4)}),
    ("fwd", 99, 1248, 10656, 0, L.LRQ_FMT_FP8, {(1, 3), (1, 4)}),
    ("bwd", 66, 8696, 768, 32, L.LRQ_FMT_INT4, {(1, 3), (1, 4), (2, 7)}),
]


@pytest.mark.parametrize("what,m,n,k,r,fmt,fast", MEASURED)
def test_plan_is_near_the_fastest_measured(what, m, n, k, r, fmt, fast):
    p = D.debug_plan(what, m, n, k, r, fmt)
    assert (p["kernel"], p["ranges"]) in fast
