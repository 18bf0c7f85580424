"""The one-pass blocked layout and the one-pass fp8 rows at the sizes where
they can go wrong: rows, columns and groups off the workgroup's 64 x 256 (or
128) columns, rows at and past the register limit, and values that a
quotient without a division could lose (signed zeros, NaN, infinities,
subnormals, ties)."""

import numpy as np
import pytest
import torch

import oracle as O
from loractl_amd import device as D

pytestmark = pytest.mark.gpu


def _blocked(q, NB, KB, pad):
    """[n, k] values in 64 x 64 blocks [NB, KB, 64, 64], padded with ``pad``."""
    n, k = q.shape
    full = np.full((NB * 64, KB * 64), pad, q.dtype)
    full[:n, :k] = q
    return full.reshape(NB, 64, KB, 64).transpose(0, 2, 1, 3)


def _nibbles(u):
    return (u[..., 0::2] | (u[..., 1::2] << 4)).astype(np.uint8)


@pytest.mark.parametrize("fmt", ["int4", "int8", "fp8"])
@pytest.mark.parametrize("n,k,g", [(1, 32, 32), (64, 64, 64), (65, 96, 32), (200, 288, 32), (130, 1024, 512),
                                   (72, 2048, 2048), (8, 4160, 64)])
def test_blocked_layout(cuda, n, k, g, fmt):
    """Both sections and both scale tables, byte for byte, from the layout's
    definition in the C header."""
    w = torch.randn(n, k, device=cuda, generator=torch.Generator(device=cuda).manual_seed(n + k))
    rows = D.quantize_int4(w, g) if fmt == "int4" else D.quantize_int8(w, g) if fmt == "int8" else D.quantize_fp8(w, True)
    b = D.block(rows)
    NB, KB = -(-n // 64), -(-k // 64)
    data = rows.data.cpu().numpy()
    if fmt == "int4":
        u = np.stack([data & 15, data >> 4], -1).reshape(n, k)
        first = _nibbles(_blocked(u, NB, KB, 8)).reshape(-1)
        second = _nibbles(_blocked(((u.astype(np.int64) - 8) & 15).T.astype(np.uint8), KB, NB, 0)).reshape(-1)
    else:
        u = data.view(np.uint8)
        first, second = _blocked(u, NB, KB, 0).reshape(-1), _blocked(u.T, KB, NB, 0).reshape(-1)
    assert np.array_equal(b.data.cpu().numpy(), np.concatenate([first, second]))
    if fmt != "fp8":
        s = np.zeros((NB * 64, KB * 64 // g), np.float32)
        s[:n, :k // g] = rows.scales.cpu().numpy()
        want = np.concatenate([s.reshape(NB, 64, -1).transpose(0, 2, 1).reshape(-1), s.T.reshape(-1)])
        assert np.array_equal(b.scales.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("per_channel", [True, False])
@pytest.mark.parametrize("n,k", [(3, 4), (5, 2048), (4, 2052), (3, 4100), (2, 16384), (2, 16388)])
def test_fp8_rows_bit_exact(cuda, n, k, per_channel):
    """Bytes and scales equal the oracle's for random rows and for rows of
    exact ties, signed zeros, subnormals and tiny values."""
    g = np.random.Generator(np.random.PCG64(n * k))
    w = (g.standard_normal((n, k)) * np.exp(g.uniform(-12, 3, (n, k)))).astype(np.float32)
    w[0, :4] = [448.0, -0.0, 2.0**-10, -2.0**-149]
    if k >= 64:
        codes = np.arange(0x7E, dtype=np.int64)
        lut = O.fp8_lut()
        w[1] = 0.0
        w[1, 0] = 448.0  # scale 1
        mid = ((lut[codes[:-1]].astype(np.float64) + lut[codes[1:]]) / 2).astype(np.float32)
        m = min(len(mid), k // 4)
        w[1, 1:1 + m] = mid[:m]
        w[1, 1 + m:1 + 2 * m] = -np.nextafter(mid[:m], np.float32(0))
        w[1, 1 + 2 * m:1 + 3 * m] = np.nextafter(mid[:m], np.float32(np.inf))
    q = D.quantize_fp8(torch.from_numpy(w).to(cuda), per_channel)
    data, scales = O.fp8_quantize(w, per_channel)
    assert np.array_equal(q.scales.cpu().numpy().view(np.uint32), np.asarray(scales, np.float32).reshape(-1).view(np.uint32))
    assert np.array_equal(q.data.cpu().numpy(), data)


def test_fp8_rows_not_finite(cuda):
    """A NaN value keeps its sign and leaves its row's scale alone; a row with
    an infinity has an infinite scale, finite values of it a signed zero."""
    w = torch.ones(3, 64, device=cuda)
    w[0, 1] = float("nan")
    w[0, 2] = -0.0
    w[1, 3] = float("inf")
    w[1, 4] = -1.0
    w[2] = 0.0
    q = D.quantize_fp8(w, True)
    d, s = q.data.cpu().numpy(), q.scales.cpu().numpy()
    assert d[0, 1] & 0x7F == 0x7F and d[0, 2] == 0x80 and d[0, 0] == 0x7E
    assert np.isinf(s[1]) and d[1, 3] & 0x7F == 0x7F and d[1, 4] == 0x80 and d[1, 0] == 0
    assert s[2] == np.float32(1e-12) and not d[2].any()
