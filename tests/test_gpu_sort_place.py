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
