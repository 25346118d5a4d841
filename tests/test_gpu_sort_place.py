"""The expert sort's last two passes in one launch, at both sides of the lines that choose it (256 chunks of 512 slots, 64 experts) and
where blocks and chunks are cut: bit for bit numpy's stable argsort.  One expert with everything, experts with nothing."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,E", [(8193, 1), (8193, 64), (8193, 65), (8704, 17), (8705, 40), (131072, 64), (131073, 64), (131072, 65),
                                 (262144, 3), (524288, 40), (65535, 33)])
@pytest.mark.parametrize("load", ["even", "one", "skewed"])
def test_place(device, L, E, load):
    from dolomite_engine_amd import ops

    rng = np.random.default_rng(L + E)
    ids = {"even": rng.integers(0, E, L), "one": np.full(L, E - 1), "skewed": (E * rng.random(L) ** 4).astype(np.int64)}[load]
    print(f"sort place L={L} E={E} {load}", flush=True)
    se, ss, off = ops.sort_bin(torch.from_numpy(ids).int().view(L, 1).to(device), E)
    order = np.argsort(ids, kind="stable")
    assert np.array_equal(ss.cpu().numpy(), order) and np.array_equal(se.cpu().numpy(), ids[order])
    assert np.array_equal(off.cpu().numpy(), np.bincount(ids, minlength=E).cumsum())


@pytest.mark.parametrize("T,E,k", [(1025, 40, 8), (2064, 64, 4), (4097, 32, 8), (32768, 40, 8), (32769, 8, 2)])
def test_behind_the_router(device, T, E, k):
    from dolomite_engine_amd import ops

    torch.manual_seed(T)
    x, w = torch.randn(T, 128, device=device).bfloat16(), torch.randn(E, 128, device=device).bfloat16()
    _, _, idx, se, ss, off = ops.router_fused_sort(x, w, k)
    for got, want in zip((se, ss, off), ops.sort_bin(idx, E)):
        assert torch.equal(got, want)
    order = np.argsort(idx.cpu().numpy().reshape(-1), kind="stable")
    assert np.array_equal(ss.cpu().numpy(), order)


@pytest.mark.parametrize("T,H,E,k", [(256, 128, 40, 8), (257, 128, 40, 8), (1025, 1024, 32, 2), (4097, 256, 40, 8), (9000, 64, 64, 1),
                                     (16400, 128, 8, 2), (33000, 64, 17, 3)])
def test_behind_the_norm(device, T, H, E, k):
    """The layer's one-call forward, whose RMSNorm router counts for the sort, against the stages, which sort by themselves."""
    from dolomite_engine_amd import Kernel, MoE, enable_kernels

    torch.manual_seed(T)
    m = MoE(hidden_size=H, intermediate_size=64, shared_intermediate_size=None, num_experts=E, num_experts_per_tok=k,
            activation_function="swiglu", add_bias=False, dropout=0.0, init_method="normal", initializer_range=0.1, m_width=None,
            num_layers=1, use_padding_free_transformer=True).to(device).bfloat16().eval()
    x = torch.randn(T, H, device=device).bfloat16()
    norm = (1 + 0.1 * torch.randn(H, device=device)).bfloat16()
    with torch.no_grad(), enable_kernels([Kernel.scattermoe]):
        got = m(x, pre_norm=(norm, 1e-5))
        stage, m._route = m._route, lambda *a, **kw: stage(*a, **kw)  # (a replaced stage: stage by stage)
        want = m(x, pre_norm=(norm, 1e-5))
    assert torch.equal(got, want)
