"""How calls plan their kernel and workspace, through the host-only planner
hook (no GPU)."""

import itertools
import random

import pytest

from loractl_amd import _lib as L
from loractl_amd import device as D

SCRATCH = L.LRQ_NOALLOC_SCRATCH_BYTES - (64 << 10)  # past the arrival counters
TOKENS = [17, 96, 192, 320, 512, 640, 896, 1024, 1792, 2112, 4096, 8192]
DIMS = [512, 2560, 3072, 4096, 9216, 12288, 14336, 16384, 18432]


@pytest.mark.parametrize("m,k,n,r", [(96, 15360, 12288, 64), (128, 18432, 12288, 64), (320, 16384, 16384, 16),
                                     (512, 15360, 3072, 32), (640, 16384, 9728, 16), (1024, 16384, 9216, 16),
                                     (2112, 14336, 4096, 16), (8192, 12288, 2560, 32), (8192, 12288, 9216, 32)])
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
                need = max(D.debug_plan(w, q, n, k, r)["bytes"] for w in ("fwd", "bwd"))
                assert need <= have, (m, q, r, need, have)
