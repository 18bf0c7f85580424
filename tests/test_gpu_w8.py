"""The 128-token tiles of 128 and 256 rows (lrq_gemm_w8.hip) at the sizes
where they can go wrong: token counts and outputs one off a tile, depths
that end inside a stage or a block, depth ranges, and factor slices that take
several rounds of workgroups."""

import pytest
import torch

import oracle as O
from gpu_helpers import case_inputs, check, gemm_path, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [(127, 224, 136, 32), (129, 256, 264, 64), (300, 1120, 520, 32), (513, 96, 1032, 32)]


def _weight(D, w, fmt, g, dev):
    wt = torch.from_numpy(w).to(dev)
    q = D.quantize_int4(wt, g) if fmt == "int4" else D.quantize_int8(wt, g) if fmt == "int8" else D.quantize_fp8(wt, True)
    return D.compute_weight(q)


@pytest.mark.parametrize("r", [8, 32, 48])
@pytest.mark.parametrize("path", ["mid128", "mid256", "mid128s", "mid256s"])
@pytest.mark.parametrize("fmt", ["int4", "int8", "fp8"])
@pytest.mark.parametrize("M,K,N,g", SHAPES)
def test_w8_tiles_against_oracle(cuda, M, K, N, g, fmt, path, r):
    """y, t, dx, dA, dB and the plain product and input gradient against the
    f64 oracle (bf16 tolerance), twice, bit for bit the same."""
    from loractl_amd import device as D

    w, x, a, b, dy = case_inputs(M, K, N, r, seed=M + N + r)
    wq = _weight(D, w, fmt, g, cuda)
    wdq = D.dequant(wq).cpu().numpy()
    xd, ad, bd, dyd = (to_dev(v, cuda) for v in (x, a, b, dy))

    def run():
        y, t = D.lora_fwd(xd, wq, ad, bd, 0.75)
        return (y, t) + tuple(D.lora_bwd(xd, dyd, wq, ad, bd, 0.75, t)) + (
            D.quant_matmul_t(xd, wq), D.quant_matmul_t_bwd(dyd, wq))

    with gemm_path(path):
        got, again = run(), run()
    for u, v in zip(got, again):
        assert torch.equal(u, v)
    y, t = O.linear_fwd(x, wdq, a, b, 0.75)
    refs = (y, t) + tuple(O.linear_bwd(x, wdq, a, b, 0.75, dy))
    refs += (O.linear_fwd(x, wdq)[0], O.linear_bwd(x, wdq, None, None, 1.0, dy)[0])
    for name, u, v in zip(("y", "t", "dx", "dA", "dB", "y base", "dx base"), got, refs):
        check(name, u, v)


@pytest.mark.parametrize("path", ["mid128s", "mid256s", "planned"])
def test_factor_slices_in_rounds(cuda, path):
    """More factor slices than the CUs beside the tiles take at once (512
    tokens, 12288 deep): every workgroup takes several, and each 64-token
    group's sum is complete before its tiles read it."""
    from loractl_amd import device as D

    M, K, N, r = 512, 12288, 3072, 32
    g = torch.Generator(device=cuda).manual_seed(5)
    w = torch.randn(N, K, device=cuda, generator=g) * 0.02
    wq = D.compute_weight(D.quantize_int4(w, 64))
    x = torch.randn(M, K, device=cuda, generator=g).to(torch.bfloat16)
    a = (torch.randn(K, r, device=cuda, generator=g) * 0.01).to(torch.bfloat16)
    b = torch.randn(r, N, device=cuda, generator=g).to(torch.bfloat16)
    with gemm_path(path):
        y, t = D.lora_fwd(x, wq, a, b, 1.0)
        y2, t2 = D.lora_fwd(x, wq, a, b, 1.0)
    D.sync()
    assert torch.equal(y, y2) and torch.equal(t, t2)
    t_ref = x.float() @ a.float()
    check("t", t, t_ref.cpu().numpy())
    check("y", y, (x.float() @ D.dequant(wq).t() + t_ref @ b.float()).cpu().numpy())


@pytest.mark.parametrize("path", ["mid64s", "mid128s", "mid256s", "mid64x128s"])
@pytest.mark.parametrize("fmt", ["int4", "fp8"])
def test_depth_ranges_of_more_tiles_than_cus(cuda, path, fmt):
    """Forced ranges where the tiles alone fill the CUs: ranges of a tile run
    in different rounds, and the last to arrive sums them all."""
    from loractl_amd import device as D

    M, K, N, r = 1100, 4096, 4096, 16
    g = torch.Generator(device=cuda).manual_seed(9)
    w = torch.randn(N, K, device=cuda, generator=g) * 0.02
    wq = D.compute_weight(D.quantize_int4(w, 64) if fmt == "int4" else D.quantize_fp8(w, True))
    bf = torch.bfloat16
    x, dy = (torch.randn(M, d, device=cuda, generator=g).to(bf) for d in (K, N))
    a = (torch.randn(K, r, device=cuda, generator=g) * 0.01).to(bf)
    b = (torch.randn(r, N, device=cuda, generator=g) * 0.1).to(bf)

    def run():
        y, t = D.lora_fwd(x, wq, a, b, 1.0)
        return (y, t) + tuple(D.lora_bwd(x, dy, wq, a, b, 1.0, t))

    with gemm_path(path):
        got, again = run(), run()
        plan = D.debug_plan("bwd", M, N, K, r, wq.fmt)
    rows = {1: 64, 2: 128, 3: 256, 4: 64}[plan["kernel"]]
    assert plan["ranges"] > 1 and plan["folded"]
    assert -(-M // (64 if path == "mid64s" else 128)) * -(-K // rows) * plan["ranges"] > 256 * (2 if rows == 64 else 1)
    for u, v in zip(got, again):
        assert torch.equal(u, v)
    W, xf, dyf, af, bff = D.dequant(wq), x.float(), dy.float(), a.float(), b.float()
    t, u = xf @ af, dyf @ bff.t()
    refs = (xf @ W.t() + t @ bff, t, dyf @ W + u @ af.t(), xf.t() @ u, t.t() @ dyf)
    for name, v, ref in zip(("y", "t", "dx", "dA", "dB"), got, refs):
        check(name, v, ref.cpu().numpy())
