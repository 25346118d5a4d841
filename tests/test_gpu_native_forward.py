"""The eval-mode forward behind one library call against the stage-by-stage calls it stands for: the same kernels on the
same inputs in the same order, so the results are equal bit for bit.  (An installed stage timer makes the module run its
stages one by one.)"""

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Timer:
    def __init__(self):
        self.stages = []

    def begin(self, name):
        self.stages.append(name)

    def end(self, name):
        pass


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,E,k,I,shared,fp8,norm,tail", [
    (1, 1536, 40, 8, 512, None, False, True, True), (64, 1024, 32, 8, 512, None, False, False, False),
    (1, 64, 4, 1, 32, 16, False, False, True), (333, 920, 17, 4, 520, 344, False, False, False),
    (700, 256, 8, 2, 512, 64, False, True, False), (40, 512, 64, 6, 256, None, True, False, True),
    (900, 512, 8, 2, 384, None, True, False, False), (50, 256, 130, 4, 64, None, False, False, False),
    (2000, 256, 8, 2, 128, None, True, False, False),  # so many rows per expert that the fp8 weights are widened
])
def test_native_forward_equals_stages(device, dtype, T, H, E, k, I, shared, fp8, norm, tail):
    from dolomite_engine_amd import Kernel, MoE, enable_kernels, ops

    if fp8 and dtype == torch.float32:
        pytest.skip("fp8 weights go with 16-bit activations")
    torch.manual_seed(T + H)
    m = MoE(hidden_size=H, intermediate_size=I, shared_intermediate_size=shared, num_experts=E, num_experts_per_tok=k,
            activation_function="swiglu", add_bias=False, dropout=0.0, init_method="normal", initializer_range=0.05,
            m_width=None, num_layers=1, use_padding_free_transformer=True).to(dtype).to(device).eval()
    if fp8:
        m.quantize_expert_weights_fp8()
    x = torch.randn(T, H, device=device, dtype=dtype)
    kwargs = {}
    if norm:
        kwargs["pre_norm"] = (1 + 0.1 * torch.randn(H, device=device, dtype=dtype), 1e-5)
    if tail:
        kwargs.update(residual=torch.randn(T, H, device=device, dtype=dtype), residual_scale=0.22)
    timer = _Timer()
    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        native = m(x, **kwargs)
        ops.set_stage_timer(timer)
        try:
            stages = m(x, **kwargs)
        finally:
            ops.set_stage_timer(None)
        again = m(x, **kwargs)
    assert timer.stages, "the second forward was meant to run stage by stage"
    assert torch.equal(native, stages)
    assert torch.equal(native, again)


def test_native_forward_refuses_what_does_not_fit(device):
    """The one-call forward takes pointers: operands whose shapes do not fit together go to the stage-by-stage code, which
    raises, and a forward hook on the down-projection still runs."""
    from dolomite_engine_amd import Kernel, MoE, enable_kernels

    def layer():
        return MoE(hidden_size=128, intermediate_size=64, shared_intermediate_size=32, num_experts=4, num_experts_per_tok=2,
                   activation_function="swiglu", add_bias=False, dropout=0.0, init_method="normal", initializer_range=0.05,
                   m_width=None, num_layers=1, use_padding_free_transformer=True).bfloat16().to(device).eval()

    x = torch.randn(9, 128, device=device, dtype=torch.bfloat16)
    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        for name, width in (("c_fc", 64), ("c_proj", 32), ("c_proj_shared", 16)):
            m = layer()
            sub = getattr(m, name)
            sub.weight = torch.nn.Parameter(sub.weight.detach()[..., :width].contiguous())
            with pytest.raises(ValueError):
                m(x)
        m = layer()
        seen = []
        want = m(x)
        m.c_proj.register_forward_hook(lambda *a: seen.append(1))
        assert torch.equal(m(x), want) and seen


def _layer(device, **kwargs):
    from dolomite_engine_amd import MoE

    sizes = dict(hidden_size=128, intermediate_size=64, shared_intermediate_size=32, num_experts=4, num_experts_per_tok=2)
    return MoE(**{**sizes, **kwargs}, activation_function="swiglu", add_bias=False, dropout=0.0, init_method="normal",
                        initializer_range=0.05, m_width=None, num_layers=1,
                        use_padding_free_transformer=True).bfloat16().to(device).eval()


@pytest.mark.parametrize("stage", ["_compute_experts", "_compute_shared_experts", "_route", "c_proj.forward",
                                   "dropout.forward"])
@pytest.mark.parametrize("where", ["subclass", "class", "instance"])
def test_native_forward_leaves_replaced_stages_alone(device, monkeypatch, stage, where):
    """A stage that a subclass or a caller replaced is called in eval() as it is in train()."""
    from dolomite_engine_amd import Kernel, MoE, enable_kernels

    torch.manual_seed(5)
    x = torch.randn(300, 128, device=device, dtype=torch.bfloat16)
    m = _layer(device, num_experts=72)  # (up to 64, the router and the sort are one call and _route is not called)
    owner = m
    *path, name = stage.split(".")
    for part in path:
        owner = getattr(owner, part)
    original = getattr(type(owner), name)
    seen = []

    def replacement(self, *args, **kwargs):
        seen.append(1)
        return original(self, *args, **kwargs)

    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        want = m(x)
        if where == "subclass":
            owner.__class__ = type("Replaced", (type(owner),), {name: replacement})
        elif where == "class":
            monkeypatch.setattr(type(owner), name, replacement)
        else:
            owner.__dict__[name] = replacement.__get__(owner)
        assert torch.equal(m(x), want)
    assert seen


@pytest.mark.parametrize("module", ["c_proj", "dropout", None])
@pytest.mark.parametrize("pre", [False, True])
def test_native_forward_leaves_hooks_alone(device, module, pre):
    """Hooks on the modules that the stages call, and hooks on every module, run in eval() too."""
    from dolomite_engine_amd import Kernel, enable_kernels

    torch.manual_seed(6)
    x = torch.randn(9, 128, device=device, dtype=torch.bfloat16)
    m = _layer(device)
    seen = []
    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        want = m(x)
        if module is not None:
            register = getattr(getattr(m, module), "register_forward_pre_hook" if pre else "register_forward_hook")
        else:
            hooks = torch.nn.modules.module
            register = hooks.register_module_forward_pre_hook if pre else hooks.register_module_forward_hook
        handle = register(lambda mod, *a: seen.append(type(mod).__name__))
        try:
            assert torch.equal(m(x), want)
        finally:
            handle.remove()
    assert seen and (module is not None or "ParameterizedExperts" in seen)


@pytest.mark.parametrize("hidden,intermediate,fp8,tokens", [(132, 64, False, 9), (136, 64, False, 9), (136, 64, True, 9),
                                                            (136, 60, False, 9)])
def test_gate_runs_once_per_forward(device, hidden, intermediate, fp8, tokens):
    """Hidden sizes that no router kernel takes: torch forms the logits, once, also where the one-call forward then refuses
    the layer (hidden or intermediate size no multiple of 8, fp8 weights with a hidden size that is no multiple of 16)."""
    from dolomite_engine_amd import Kernel, enable_kernels

    torch.manual_seed(7)
    m = _layer(device, hidden_size=hidden, intermediate_size=intermediate)
    if fp8:
        m.quantize_expert_weights_fp8()
    seen = []
    m.gate.register_forward_hook(lambda *a: seen.append(1))
    x = torch.randn(tokens, hidden, device=device, dtype=torch.bfloat16)
    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        m(x)
    assert len(seen) == 1
