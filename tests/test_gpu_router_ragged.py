"""The router of rows that are a multiple of 8 but not of 16 long, at the edges of its tiles: rows that end in the middle of a lane's 16
values, of a step of 64 and of the four waves' shares; 16 tokens and 16 experts a block.

Logits against a product in 64 bits: exact operands, fp32 sums (relative error below 2^-14 of the sum of the magnitudes for 1000
terms), one rounding (2^-8 of the value in bf16, 2^-11 in fp16), two with a bias.  Selection and gates against the logits that the
kernel wrote: value descending, index ascending; an fp32 softmax and one rounding."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("T,H,E,k", [(1, 8, 1, 1), (15, 24, 16, 4), (17, 56, 17, 17), (16, 72, 64, 64), (33, 248, 33, 8),
                                     (3001, 920, 17, 4), (40, 1032, 48, 2), (5, 120, 7, 3)])
def test_router_ragged(device, dtype, bias, T, H, E, k):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(T * 31 + H)
    x, w = torch.randn(T, H, generator=g).to(dtype), (torch.randn(E, H, generator=g) * 0.1).to(dtype)
    b = torch.randn(E, generator=g) if bias else None
    print(f"router ragged T={T} H={H} E={E} k={k} {dtype} {bias}", flush=True)
    assert ops.router_ragged_supported(x, E, k)
    logits, gates, idx = ops.router_ragged(x.to(device), w.to(device), k, bias=None if b is None else b.to(device), return_logits=True)
    none, gates2, idx2 = ops.router_ragged(x.to(device), w.to(device), k, bias=None if b is None else b.to(device))
    assert none is None and torch.equal(gates, gates2) and torch.equal(idx, idx2)
    want = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = eps * want.abs() + 2.0 ** -14 * size
    if bias:
        want = want + b.double()
        bound = bound + eps * want.abs()
    assert ((logits.cpu().double() - want).abs() <= bound).all()
    top = logits.cpu().float().sort(dim=1, descending=True, stable=True)
    assert torch.equal(idx.cpu().long(), top.indices[:, :k])
    torch.testing.assert_close(gates.cpu().float(), top.values[:, :k].softmax(dim=1), rtol=2 * eps, atol=2.0 ** -24)


def test_gate_that_is_more_than_its_weight_is_called(device):
    from dolomite_engine_amd import Kernel, MoE, enable_kernels

    torch.manual_seed(3)
    m = MoE(hidden_size=136, intermediate_size=64, shared_intermediate_size=None, num_experts=5, num_experts_per_tok=2,
            activation_function="swiglu", add_bias=False, dropout=0.0, init_method="normal", initializer_range=0.1, m_width=None,
            num_layers=1, use_padding_free_transformer=True).to(device).to(torch.float16).eval()
    x = torch.randn(20, 136, device=device, dtype=torch.float16)
    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        plain = m(x)
        handle = m.gate.register_forward_hook(lambda mod, args, out: -out)
        hooked = m(x)
        handle.remove()
        assert torch.equal(plain, m(x))
    assert not torch.equal(plain, hooked)
