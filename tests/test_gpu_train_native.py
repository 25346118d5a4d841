"""A training step's routed experts behind one library call in either direction against the stage-by-stage functions that it
stands for: the same products, sums and roundings in the same order on the same operands, so every result is the same bits.  With
shared experts that takes in the order in which the three gradients of x are added."""

import pytest
import torch

from dolomite_engine_amd import Kernel, MoE, enable_kernels
from dolomite_engine_amd.loss import clear_aux_loss, get_aux_loss

pytestmark = pytest.mark.gpu

SIZES = {"even": (512, 256, 16, 4, 264), "wide": (96, 1024, 8, 2, 520), "small": (5, 128, 8, 8, 64), "one": (1, 64, 8, 1, 8),
         "large": (3000, 256, 40, 8, 128), "blocks": (2049, 128, 64, 6, 64)}


def _layer(device, dtype, sizes, shared=None):
    T, H, E, k, I = sizes
    torch.manual_seed(T)
    layer = MoE(hidden_size=H, intermediate_size=I, shared_intermediate_size=shared, num_experts=E, num_experts_per_tok=k,
                activation_function="swiglu", add_bias=False, dropout=0.0, init_method="normal", initializer_range=0.1,
                m_width=None, num_layers=1, use_padding_free_transformer=True).to(device).to(dtype).train()
    return layer, torch.randn(T, H, device=device).to(dtype)


def _step(layer, x, parts="both", x_grad=True, dy_form="plain", scale=None):
    layer.zero_grad(set_to_none=True)
    x = x.detach().clone().requires_grad_(x_grad)
    clear_aux_loss()
    with enable_kernels([Kernel.scattermoe]):
        y = layer(x, **({} if scale is None else dict(residual=x, residual_scale=scale)))
        aux = get_aux_loss()
        torch.manual_seed(7)
        dy = torch.randn(*y.shape, device=y.device).to(y.dtype)
        if dy_form == "strided":
            dy = torch.stack([dy, dy], dim=-1)[..., 0]
        elif dy_form == "misaligned":
            dy = torch.cat([dy.reshape(-1)[:1], dy.reshape(-1)])[1:].view_as(dy)
        wanted = [(y, dy), (aux, torch.full_like(aux, 0.3))]
        if parts != "both":
            wanted = wanted[:1] if parts == "y" else wanted[1:]
        torch.autograd.backward(*zip(*wanted))
    out = {"y": y.detach(), "aux": aux.detach(), "x": x.grad}
    return out | {n: p.grad for n, p in layer.named_parameters()}


def _check(monkeypatch, layer, x, **how):
    taken = []
    native = MoE._train_native
    monkeypatch.setattr(MoE, "_train_native", lambda self, h: taken.append(native(self, h)) or taken[-1])
    got = _step(layer, x, **how)
    assert taken and taken[-1] is not None, "the one-call form did not run"
    monkeypatch.setattr(MoE, "_train_native", lambda self, h: None)
    want = _step(layer, x, **how)
    monkeypatch.undo()
    for name, w in want.items():
        g = got[name]
        assert (g is None) == (w is None), name
        if w is None:
            continue
        assert g.dtype == w.dtype and g.shape == w.shape, name
        assert torch.equal(g, w), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", list(SIZES))
def test_equals_stages(device, monkeypatch, name, dtype):
    layer, x = _layer(device, dtype, SIZES[name])
    print(f"train native {name} {dtype}", flush=True)
    _check(monkeypatch, layer, x)


# sizes where the experts' weight gradients are cut into groups, whose partial results lie where the backward's first operands were:
# both, with H above and below 2 I and I, the down-projection's alone, and more than 32768 slots
PLANNED = {"both": ((4097, 256, 8, 2, 520), (0, 0)), "tall": ((4097, 512, 8, 2, 136), (0, 0)), "one of them": ((1160, 256, 8, 1, 520), (1, 0)),
           "long": ((4600, 128, 64, 8, 64), (0, 0))}


@pytest.mark.parametrize("load", ["even", "skewed"])
@pytest.mark.parametrize("name", list(PLANNED))
def test_planned_weight_gradients(device, monkeypatch, name, load):
    from dolomite_engine_amd import _lib

    (T, H, E, k, I), whole = PLANNED[name]
    choose = _lib.load().mi_moe_grouped_wgrad_whole
    assert (choose(T * k, T * k, T, 2 * I, H, E), choose(T * k, T, T * k, H, I, E)) == whole
    layer, x = _layer(device, torch.bfloat16, PLANNED[name][0])
    if load == "skewed":
        layer.router_logit_bias = -2 * (torch.arange(E, device=device) + 1.0).log()
    print(f"train native planned {name} {load}", flush=True)
    _check(monkeypatch, layer, x)


@pytest.mark.parametrize("how", [dict(parts="y"), dict(parts="aux"), dict(x_grad=False), dict(parts="aux", x_grad=False),
                                 dict(dy_form="strided"), dict(scale=0.25)])
def test_parts_and_forms(device, monkeypatch, how):
    layer, x = _layer(device, torch.bfloat16, SIZES["even"])
    print(f"train native {how}", flush=True)
    _check(monkeypatch, layer, x, **how)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name,how", [("even", {}), ("even", dict(parts="y")), ("even", dict(parts="aux")), ("even", dict(x_grad=False)),
                                      ("even", dict(scale=0.25)), ("one", {}), ("large", {})])
def test_shared_experts_equal_stages(device, monkeypatch, name, how, dtype):
    layer, x = _layer(device, dtype, SIZES[name], shared=72)
    print(f"train native shared {name} {how} {dtype}", flush=True)
    _check(monkeypatch, layer, x, **how)


def test_misaligned_gradient(device):
    """(The stages refuse an upstream gradient that does not start on 16 bytes.)"""
    layer, x = _layer(device, torch.bfloat16, SIZES["even"])
    want, got = _step(layer, x), _step(layer, x, dy_form="misaligned")
    assert all(torch.equal(got[n], w) for n, w in want.items())


@pytest.mark.parametrize("frozen", [("gate",), ("c_fc",), ("c_proj",), ("c_fc", "c_proj"), ("gate", "c_fc", "c_proj")])
def test_frozen_parameters_get_no_gradient(device, frozen):
    layer, x = _layer(device, torch.bfloat16, SIZES["even"], shared=64)
    full = _step(layer, x)
    for name in frozen:
        getattr(layer, name).weight.requires_grad_(False)
    part = _step(layer, x)
    for name, g in part.items():
        if name.split(".")[0] in frozen:
            assert g is None, name
        else:
            assert torch.equal(g, full[name]), name


def test_router_without_a_gradient_leaves_the_loss_without_one(device):
    layer, x = _layer(device, torch.bfloat16, SIZES["even"])
    layer.gate.weight.requires_grad_(False)
    clear_aux_loss()
    with enable_kernels([Kernel.scattermoe]):
        y = layer(x)
    assert y.requires_grad and not get_aux_loss().requires_grad


@pytest.mark.parametrize("hook", ["full_backward_hook", "full_backward_pre_hook"])
@pytest.mark.parametrize("everywhere", [False, True])
def test_backward_hooks_are_called(device, hook, everywhere):
    layer, x = _layer(device, torch.bfloat16, SIZES["even"])
    want = _step(layer, x)
    calls = []
    call = lambda mod, *grads: calls.append(mod) if mod is layer.dropout else None
    handle = (getattr(torch.nn.modules.module, "register_module_" + hook)(call) if everywhere
              else getattr(layer.dropout, "register_" + hook)(call))
    try:
        got = _step(layer, x)
    finally:
        handle.remove()
    assert len(calls) == 2  # behind the experts and in front of the residual
    assert all(torch.equal(got[n], w) for n, w in want.items())


def _strided(t):
    return torch.stack([t, t], dim=-1)[..., 0]


def _shifted(t):
    return torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape)


@pytest.mark.parametrize("unpack", [_strided, _shifted, lambda t: t.transpose(0, -1).contiguous().transpose(0, -1), lambda t: t.to("cuda:0")])
def test_saved_tensor_hooks(device, unpack):
    """What a hook hands back has the values, but not the strides or the alignment of what it was given."""
    layer, x = _layer(device, torch.bfloat16, SIZES["wide"])
    want = _step(layer, x)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu(), lambda t: unpack(t.to(device))):
        got = _step(layer, x)
    assert packed and all(torch.equal(got[n], w) for n, w in want.items())


def test_parametrized_weight_is_computed_once(device):
    layer, x = _layer(device, torch.bfloat16, SIZES["even"])
    want = _step(layer, x)
    calls = []

    class Counted(torch.nn.Module):
        def forward(self, w):
            calls.append(1)
            return w * 1

    torch.nn.utils.parametrize.register_parametrization(layer.c_fc, "weight", Counted())
    calls.clear()
    got = _step(layer, x)
    assert len(calls) == 1
    assert torch.equal(got["y"], want["y"]) and torch.equal(got["c_fc.parametrizations.weight.original"], want["c_fc.weight"])


def test_replaced_stage_is_called(device):
    layer, x = _layer(device, torch.bfloat16, SIZES["even"])
    calls = []
    compute = layer._compute_experts
    layer._compute_experts = lambda *a, **k: calls.append(1) or compute(*a, **k)
    _step(layer, x)
    assert calls
