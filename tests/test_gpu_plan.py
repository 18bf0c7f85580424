"""How calls plan their kernel: once, and within the limits of the call and of
the launch."""

import pytest
import torch

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
