"""The router's form for at most a group of 16 tokens per CU (every load requested at once, up to 16 tokens with the sort behind it):
tokens at the edges of a group and of the rules, hidden sizes at the edges of a lane's 16 values, a K step, a wave's turn and the
limit of 2048, experts at the edges of a block of 16."""

import pytest
import torch

from oracle import moe_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 321, 4096, 4097])
@pytest.mark.parametrize("H,E,k", [(16, 1, 1), (48, 16, 8), (64, 17, 2), (512, 40, 8), (528, 64, 6), (1040, 33, 3), (2032, 16, 8), (2032, 32, 8),
                                   (2048, 33, 8), (2064, 16, 4)])
@pytest.mark.parametrize("gamma", ["none", "aligned", "odd"])
def test_router_direct(device, dtype, T, H, E, k, gamma):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(T * 5 + H + E)
    h = torch.randn(T, H, generator=g).to(dtype)
    w = (torch.randn(E, H, generator=g) * 0.05).to(dtype)
    b = torch.randn(E, generator=g) if E % 2 else None
    ln = None if gamma == "none" else (1 + 0.1 * torch.randn(H + 1, generator=g)).to(dtype)[1:]
    print(f"router direct T={T} H={H} E={E} k={k} {dtype} gamma={gamma}", flush=True)
    ln_dev = None
    if ln is not None:
        ln_dev = torch.empty(H + 8, dtype=dtype, device=device)[1 if gamma == "odd" else 0:][:H].copy_(ln)
    hd, wd, bd = h.to(device), w.to(device), None if b is None else b.to(device)
    xn, logits, gates, idx = ops.rmsnorm_router_fused(hd, ln_dev, 1e-5, wd, k, bias=bd, return_logits=True)
    # one rounding of the fp32 norm, and a rounding boundary crossed by its own error: two units at most
    h32 = h.double()
    want = h32 * (h32.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * (1.0 if ln is None else ln.double())
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    torch.testing.assert_close(xn.cpu().double(), want, rtol=unit, atol=2.0 ** -24)
    # the routing is the routing of that norm: fp32 sums, one rounding (with a bias a second one, of the product)
    product = xn.cpu().float() @ w.float().t()
    ref = product if b is None else product + b
    room = unit * (ref.abs() + (0 if b is None else product.abs())) + 2.0 ** -20 * H ** 0.5
    assert bool(((logits.cpu().float() - ref).abs() <= room).all())
    vals, ref_idx = oracle.topk_canonical(logits.cpu(), k)
    assert torch.equal(idx.cpu().long(), ref_idx)
    ulp = gates.cpu().view(torch.int16).int() - oracle.softmax_topk(vals, dtype).view(torch.int16).int()
    assert ulp.abs().max() <= 1
    # without the norm: the same sums in the same order wherever both calls run this form
    plain = ops.router_fused(xn, wd, k, bias=bd, return_logits=True)
    if T > 320 or (T <= 16 and H <= 2048 and (T + E) * H <= 65536):
        if H <= 2048:
            assert all(torch.equal(p, q) for p, q in zip(plain, (logits, gates, idx)))
        one_launch = ops.router_fused(xn, wd, k, bias=bd, return_logits=True, split_k=False)
        assert all(torch.equal(p, q) for p, q in zip(one_launch, plain))
    # with the sort
    if ops.router_fused_sort_supported(xn, E, k):
        got = ops.router_fused_sort(xn, wd, k, bias=bd, return_logits=True)
        assert all(torch.equal(p, q) for p, q in zip(got[:3], plain))
        rse, rss, roff = oracle.sort_bin(got[2].cpu(), E)
        assert [torch.equal(p.cpu().long(), q) for p, q in zip(got[3:], (rse, rss, roff))] == [True] * 3


@pytest.mark.parametrize("T", [1, 16, 17])
@pytest.mark.parametrize("H,E,k", [(48, 4, 1), (1536, 40, 8), (2048, 33, 8), (2064, 33, 2)])
def test_layer_with_norm_sorts_in_the_router(device, T, H, E, k):
    """The one-call forward of the block's form against its stages one by one: equal bit for bit."""
    from dolomite_engine_amd import Kernel, MoE, enable_kernels, ops

    class Timer:
        def begin(self, name):
            pass

        def end(self, name):
            pass

    torch.manual_seed(T + H)
    m = MoE(hidden_size=H, intermediate_size=64, shared_intermediate_size=None, num_experts=E, num_experts_per_tok=k,
            activation_function="swiglu", add_bias=False, dropout=0.0, init_method="normal", initializer_range=0.05, m_width=None,
            num_layers=1, use_padding_free_transformer=True).bfloat16().to(device).eval()
    x = torch.randn(T, H, device=device, dtype=torch.bfloat16)
    norm = (1 + 0.1 * torch.randn(H, device=device)).bfloat16()
    print(f"layer with norm T={T} H={H} E={E} k={k}", flush=True)
    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        native = [m(x, pre_norm=(norm, 1e-5)) for _ in range(3)]
        ops.set_stage_timer(Timer())
        try:
            stages = m(x, pre_norm=(norm, 1e-5))
        finally:
            ops.set_stage_timer(None)
    assert all(torch.equal(y, stages) for y in native)
