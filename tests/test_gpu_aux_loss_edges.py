"""The aux loss where its rows per wave and columns per lane end: one row to just over a block of 32, 1, 64, 65 and 256
experts, more than 64 chosen experts.  Against the definition in float64: fp32 sums of at most 100 rows and 256 experts, hardware
exp and log of a few units in the last place."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 3, 5, 29, 31, 32, 33, 100])
@pytest.mark.parametrize("E,k", [(1, 1), (17, 2), (64, 8), (65, 65), (129, 4), (256, 100)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_aux_loss_edges(device, T, E, k, dtype):
    from dolomite_engine_amd import ops

    print(f"aux loss T={T} E={E} k={k} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T * 1000 + E)
    logits = (2 * torch.randn(T, E, generator=g)).to(dtype)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).int()
    loss = ops.aux_loss(logits.to(device), idx.to(device))[0]
    x = logits.double()
    A, f = x.softmax(-1).sum(0), torch.bincount(idx.flatten().long(), minlength=E).double()
    want = E * (A / A.sum() * f / f.sum()).sum() + 0.1 * (x.logsumexp(-1) ** 2).mean()
    torch.testing.assert_close(loss.double().cpu(), want, rtol=2e-5, atol=2e-6)
