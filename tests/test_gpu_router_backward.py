"""The router's backward when a gradient reaches only one of its outputs (none is filled in for the other), and its input
gradient from the gate weight as it lies: expert counts that the transposed-weight GEMM takes (multiples of 8) and that go
through a transposed copy, against the gradient of the same function in float64.  d logits is rounded to the model dtype
once (2^-9 relative in bf16), the products once more; 2^-6 of the largest entry bounds both with room for the sums."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,k", [(1, 64, 8, 2), (509, 1024, 32, 8), (77, 48, 40, 4), (300, 256, 17, 3), (130, 72, 24, 8)])
@pytest.mark.parametrize("which", ["logits", "gates", "both"])
def test_router_backward_partial_gradients(device, T, H, E, k, which):
    from dolomite_engine_amd.autograd import FusedRouter
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(T + E)
    x = torch.randn(T, H, generator=g).bfloat16().to(device).requires_grad_(True)
    w = (torch.randn(E, H, generator=g) * 0.1).bfloat16().to(device).requires_grad_(True)
    if not ops.router_fused_supported(x, E, k):
        pytest.skip("not a shape of the fused router")
    logits, gates, experts, *_ = FusedRouter.apply(x, w, None, k)
    dl = torch.randn(T, E, generator=g).bfloat16().to(device)
    dg = torch.randn(T, k, generator=g).bfloat16().to(device)
    outs, grads = zip(*[p for p in ((logits, dl), (gates, dg)) if which in ("both", "logits" if p[0] is logits else "gates")])
    torch.autograd.backward(outs, grads)

    x64, w64 = (t.detach().double().requires_grad_(True) for t in (x, w))
    l64 = x64 @ w64.t()
    g64 = torch.softmax(l64.gather(1, experts.long()), dim=1)
    outs = [o for o, n in ((l64, "logits"), (g64, "gates")) if which in ("both", n)]
    torch.autograd.backward(outs, [t.double() for t in grads])
    for got, want in ((x.grad, x64.grad), (w.grad, w64.grad)):
        assert (got.double() - want).abs().max() <= 2.0 ** -6 * want.abs().max()
