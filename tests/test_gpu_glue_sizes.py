"""The block glue's gradients where their row loop, their register sets and
their column sums can go wrong: row counts around the four wavefronts of a
workgroup and the 256 workgroups, every width class up to 4096; and the
rotation tables at odd sizes."""

import math

import numpy as np
import pytest
import torch

from loractl_amd.mmdit_ops import gated_residual, modnorm, rope_tables

pytestmark = pytest.mark.gpu


def _close(got, ref, name, terms=1):
    # one bf16 rounding (2^-8 of the value) plus f32 sums of `terms` products
    err = (got.double() - ref).abs()
    bound = 2.0**-8 * ref.abs() + 2.0**-20 * math.sqrt(terms) * ref.abs().max()
    assert bool((err <= bound).all()), f"{name}: {float((err - bound).max())}"


@pytest.mark.parametrize("rows", [1, 5, 257, 1030, 2051])
@pytest.mark.parametrize("h", [8, 520, 1536, 2056, 3072, 3584, 4096])
def test_gradients_match_f64(cuda, rows, h):
    g = torch.Generator(device=cuda).manual_seed(rows + h)
    bf = torch.bfloat16
    x, o, dy = (torch.randn(rows, h, device=cuda, generator=g).to(bf) for _ in range(3))
    v = [torch.randn(1, h, device=cuda, generator=g).to(bf) for _ in range(3)]
    ins = [t.clone().requires_grad_() for t in (x, o, *v)]
    f64 = [t.double().requires_grad_() for t in (x, o, *v)]
    a, b = modnorm(ins[0], ins[2], ins[3]), gated_residual(ins[0], ins[4], ins[1])
    n = f64[0] * torch.rsqrt(f64[0].square().mean(-1, keepdim=True) + 1e-5)
    ra, rb = (f64[2] + 1) * n + f64[3], f64[0] + f64[4] * f64[1]
    _close(a, ra.detach(), "modnorm")
    _close(b, rb.detach(), "gated residual")
    for name, got, ref, idx in (("modnorm", a, ra, (0, 2, 3)), ("gated residual", b, rb, (4, 1))):
        gg = torch.autograd.grad(got, [ins[i] for i in idx], dy, retain_graph=True)
        again = torch.autograd.grad(got, [ins[i] for i in idx], dy)
        rr = torch.autograd.grad(ref, [f64[i] for i in idx], dy.double())
        for i, u, w, r in zip(idx, gg, again, rr):
            assert torch.equal(u, w)
            _close(u, r, f"d {name} / d input {i}", terms=h if i == 0 else rows)


@pytest.mark.parametrize("L,hd,theta", [(1, 64, 10000.0), (333, 128, 10000.0), (4608, 128, 10000.0), (70, 2, 500.0),
                                        (0, 64, 10000.0)])
def test_rope_tables_kernel_matches_host(cuda, L, hd, theta):
    """The GPU's tables equal the host's f64 ones to one f32 rounding."""
    c, s = rope_tables(L, hd, cuda, theta)
    ch, sh = rope_tables(L, hd, "cpu", theta)
    assert c.shape == ch.shape == (L, hd // 2) and c.dtype == torch.float32
    if L:
        assert float((c.cpu() - ch).abs().max()) <= 2.0**-24 and float((s.cpu() - sh).abs().max()) <= 2.0**-24


def test_rope_tables_kernel_takes_what_the_host_takes(cuda):
    """A theta that is no Python float, and an empty head."""
    theta = np.float32(500.0)
    for got, ref in zip(rope_tables(70, 64, cuda, theta), rope_tables(70, 64, "cpu", theta)):
        assert float((got.cpu() - ref).abs().max()) <= 2.0**-24
    assert rope_tables(3, 0, cuda)[0].shape == rope_tables(3, 0, "cpu")[0].shape
    # no device (the host's), and sizes that are whole but not integers
    for got in (rope_tables(5, 64, None), rope_tables(5.0, 64.0, cuda), rope_tables(np.int64(5), np.int32(64), cuda)):
        for t, ref in zip(got, rope_tables(5, 64, "cpu")):
            assert t.shape == ref.shape and float((t.cpu() - ref).abs().max()) <= 2.0**-24
