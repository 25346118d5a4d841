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


def _layer(device, dtype, H, E, k):
    from dolomite_engine_amd import MoE

    torch.manual_seed(H)
    return MoE(hidden_size=H, intermediate_size=64, shared_intermediate_size=None, num_experts=E, num_experts_per_tok=k,
               activation_function="swiglu", add_bias=False, dropout=0.0, init_method="normal", initializer_range=0.1, m_width=None,
               num_layers=1, use_padding_free_transformer=True).to(device).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("T,H,E,k", [(1500, 920, 17, 4), (333, 1032, 64, 8), (64, 24, 8, 2)])
def test_selection_does_not_depend_on_a_gradient(device, dtype, bias, T, H, E, k):
    """Near-ties: every expert's weights are the same but for a part of about a rounding step of the logits."""
    from dolomite_engine_amd import Kernel, enable_kernels

    m = _layer(device, dtype, H, E, k)
    w = torch.randn(1, H) * 0.1
    with torch.no_grad():
        m.gate.weight.copy_(w + torch.randn(E, H) * w.norm() * torch.finfo(dtype).eps / H ** 0.5)
    if bias:
        m.router_logit_bias = (torch.randn(E) * torch.finfo(dtype).eps).to(device)
    x = torch.randn(T, H).to(dtype).to(device).requires_grad_(True)
    print(f"router ragged selection T={T} H={H} E={E} k={k} {dtype} {bias}", flush=True)
    routed = []
    with enable_kernels([Kernel.scattermoe]):
        for mode in (True, False):
            m.train(mode)
            routed.append(m._compute_routing_weights(x))
            with torch.no_grad():
                routed.append(m._compute_routing_weights(x))
    assert routed[0][0].requires_grad and routed[0][1].requires_grad
    for logits, _, experts in routed[1:]:
        assert torch.equal(logits, routed[0][0]) and torch.equal(experts, routed[0][2])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,E,k", [(300, 136, 7, 2), (17, 920, 17, 4)])
def test_gradient_of_the_logits(device, dtype, T, H, E, k):
    """Against products in 64 bits: exact operands, one rounding (2^-8 or 2^-11 of the value) and fp32 sums, or sums of rounded
    parts, which the absolute term allows for (terms of unit size, a rounding step of the largest partial sum)."""
    from dolomite_engine_amd.autograd import RaggedLogits

    g = torch.Generator().manual_seed(T)
    x, w, dl = (torch.randn(*s, generator=g).to(dtype).to(device) for s in ((T, H), (E, H), (T, E)))
    x.requires_grad_(True), w.requires_grad_(True)
    dx, dw = torch.autograd.grad(RaggedLogits.apply(x, w, None, k), (x, w), dl)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for got, a, b in ((dx, dl, w), (dw, dl.t(), x)):
        want = a.double() @ b.double()
        bound = eps * want.abs() + eps * 2.0 ** -4 * (a.double().abs() @ b.double().abs())
        assert got.dtype == dtype and ((got.double() - want).abs() <= bound).all()
    only, = torch.autograd.grad(RaggedLogits.apply(x.detach(), w, None, k), (w,), dl)
    assert torch.equal(only, dw)


@pytest.mark.parametrize("which", ["gate", "global"])
@pytest.mark.parametrize("training", [True, False])
def test_backward_hook_of_the_gate_is_called(device, which, training):
    from dolomite_engine_amd import Kernel, enable_kernels

    m = _layer(device, torch.float16, 136, 5, 2).train(training)
    x = torch.randn(20, 136, device=device, dtype=torch.float16, requires_grad=True)
    calls = []
    hook = lambda mod, *a: calls.append(mod) if mod is m.gate else None
    handle = (m.gate.register_full_backward_hook(hook) if which == "gate"
              else torch.nn.modules.module.register_module_full_backward_hook(hook))
    with enable_kernels([Kernel.scattermoe]):
        m(x).sum().backward()
    handle.remove()
    assert calls


@pytest.mark.parametrize("training", [True, False])
def test_bias_of_another_shape_is_broadcast(device, training):
    from dolomite_engine_amd import Kernel, enable_kernels, ops

    m = _layer(device, torch.bfloat16, 136, 5, 2).train(training)
    x = torch.randn(20, 136, device=device).bfloat16()
    forms = [torch.tensor(0.5), torch.tensor([0.5], device=device), torch.full((20, 5), 0.5, device=device), torch.full((5,), 0.5, device=device)]
    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        routed = []
        for bias in forms:
            m.router_logit_bias = bias
            routed.append(m._compute_routing_weights(x))
            m(x)
    for got in routed[:2]:
        assert all(torch.equal(a, b) for a, b in zip(got, routed[2]))
    torch.testing.assert_close(routed[3][0], routed[2][0], rtol=2.0 ** -7, atol=2.0 ** -7)  # (another order of summation: a rounding step)
    with pytest.raises(ValueError):
        ops.router_ragged(x, m.gate.weight.detach(), 2, bias=forms[1])


def test_bias_with_a_gradient_gets_one(device):
    from dolomite_engine_amd import Kernel, enable_kernels

    m = _layer(device, torch.bfloat16, 136, 5, 2).train()
    m.router_logit_bias = torch.zeros(5, device=device, requires_grad=True)
    with enable_kernels([Kernel.scattermoe]):
        m(torch.randn(20, 136, device=device).bfloat16()).sum().backward()
    assert m.router_logit_bias.grad is not None


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
