"""How calls plan their kernel: once, and within the limits of the call and of
the launch."""

import pytest
import torch

from gpu_helpers import check
from loractl_amd import device as D

pytestmark = pytest.mark.gpu


def _case(dev, M, K, N, r, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    wq = D.compute_weight(D.quantize_int4(torch.randn(N, K, device=dev, generator=g) * 0.02, 64))
    x = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    dy = torch.randn(M, N, device=dev, generator=g).to(torch.bfloat16)
    a = ((torch.rand(K, r, device=dev, generator=g) * 2 - 1) / K ** 0.5).to(torch.bfloat16)
    b = (torch.randn(r, N, device=dev, generator=g) * 1e-2).to(torch.bfloat16)
    return wq, x, dy, a, b


@pytest.mark.parametrize("M,r,most", [(1, 16, 0), (16, 0, 0), (256, 16, 1), (256, 0, 1), (4096, 32, 2), (300, 64, 1)])
def test_a_call_evaluates_the_cost_model_once(cuda, M, r, most):
    """Once past 16 tokens; twice where the folded kernels are ruled out first
    (the 256-token tiles at 4096 tokens); never for a few tokens."""
    K, N = 2560, 9728
    wq, x, dy, a, b = _case(cuda, M, K, N, max(r, 1), M)

    def formed():
        return D.debug_plan("fwd", 1, 8, 32, 8)["plans"]

    def calls():
        if r == 0:
            yield lambda: D.quant_matmul_t(x, wq)
            yield lambda: D.quant_matmul_t_bwd(dy, wq)
        else:
            t = torch.zeros(M, r, dtype=torch.bfloat16, device=cuda)
            yield lambda: D.lora_fwd(x, wq, a, b, 1.0)
            yield lambda: D.lora_bwd(x, dy, wq, a, b, 1.0, t)

    for call in calls():
        before = formed()
        call()
        assert formed() - before <= most


@pytest.mark.parametrize("M,K,N,r", [(64, 18432, 12288, 64), (96, 15360, 12288, 64), (512, 15360, 3072, 32),
                                     (640, 16384, 9728, 16), (1024, 14336, 2560, 32), (1024, 16384, 9216, 16),
                                     (2112, 14336, 4096, 16), (8192, 12288, 9216, 32)])
def test_noalloc_takes_a_kernel_that_fits_its_scratch(cuda, M, K, N, r):
    """Shapes whose fastest plan needs more than the 32 MiB scratch array
    (depth-range partials, t's slice partials) run on another that fits; and
    shapes just within it."""
    wq, x, _, a, b = _case(cuda, M, K, N, r, M + K)
    y = torch.empty((M, N), dtype=torch.bfloat16, device=cuda)
    t = torch.empty((M, r), dtype=torch.bfloat16, device=cuda)
    D.lora_fwd_noalloc(x, wq, a, b, 1.0, y, t)
    D.sync()
    rows = torch.linspace(0, M - 1, min(M, 64), device=cuda).long()
    xf = x[rows].float()
    t_ref = xf @ a.float()
    check("t", t[rows], t_ref.cpu().numpy())
    check("y", y[rows], (xf @ D.dequant(wq).t() + t_ref @ b.float()).cpu().numpy())


@pytest.mark.parametrize("M,N", [(100000, 21512), (100000, 18440)], ids=["past 4 GiB", "past 2 GiB"])
def test_input_gradient_of_activations_past_the_fold_offsets(cuda, M, N):
    """The side products formed beside the tiles address dy [m, n] as one
    buffer with 32-bit offsets; a larger dy takes separate launches. A NaN in
    dy (at the byte offset that masked loads use) stays in its own token."""
    K, r = 512, 16
    wq, x, dy, a, b = _case(cuda, M, K, N, r, N)
    bad = 2 ** 30 // N
    dy.view(-1)[2 ** 30] = float("nan")
    dx, da, db = D.lora_bwd(x, dy, wq, a, b, 1.0, torch.zeros(M, r, dtype=torch.bfloat16, device=cuda))
    D.sync()
    rows = torch.tensor([0, 1, bad - 1, bad + 1, M // 2, M - 1], device=cuda)
    dyf = dy[rows].float()
    check("dx", dx[rows], (dyf @ D.dequant(wq) + (dyf @ b.float().t()) @ a.float().t()).cpu().numpy())
    nan = torch.isnan(dx.float()).any(1).nonzero().flatten()
    assert nan.tolist() == [bad]


@pytest.mark.parametrize("M,m,K,N,r", [(1024, 192, 3072, 3072, 16), (4096, 896, 3072, 12288, 32)])
def test_reserve_serves_every_smaller_token_count(cuda, M, m, K, N, r):
    """After lrq_reserve for M tokens a call of m < M tokens is captured
    without allocating, although it may split its depth into more ranges."""
    wq, x, dy, a, b = _case(cuda, m, K, N, r, m)
    y, dx = torch.empty_like(dy), torch.empty_like(x)
    t = torch.empty((m, r), dtype=torch.bfloat16, device=cuda)
    da = torch.empty((K, r), device=cuda)
    db = torch.empty((r, N), device=cuda)
    stream = torch.cuda.Stream()
    ctx = D.Context(0, stream.cuda_stream)  # a context of its own: no workspace yet
    key = (0, stream.cuda_stream)
    old = D._ctxs.get(key)
    D._ctxs[key] = ctx
    try:
        stream.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            D.reserve(M, N, K, r)
            with torch.cuda.graph(graph, stream=stream):
                D.lora_fwd(x, wq, a, b, 1.0, y=y, t=t)
                D.lora_bwd(x, dy, wq, a, b, 1.0, t, out=(dx, da, db))
        graph.replay()
        torch.cuda.synchronize()
    finally:
        del graph
        if old is None:
            del D._ctxs[key]
        else:
            D._ctxs[key] = old
    y0, t0 = D.lora_fwd(x, wq, a, b, 1.0)
    for got, want in zip((y, t, dx, da, db), (y0, t0) + tuple(D.lora_bwd(x, dy, wq, a, b, 1.0, t0))):
        assert torch.equal(got, want)
