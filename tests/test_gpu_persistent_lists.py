"""Persistent grouped GEMM: the search for a tile's expert at the ends of its blocks of 64 experts, and outputs beyond what one
32-bit byte offset reaches.  Bounds as in test_gpu_persistent.py: the one rounding of the result plus the order of the fp32 sum."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = dict(rtol=2.0 ** -8, atol=2e-3)


@pytest.mark.parametrize("E", [1, 2, 63, 64, 65, 127, 128, 129, 192, 193, 256])
@pytest.mark.parametrize("empty", ["none", "ends", "block", "most"])
def test_expert_of_a_tile(device, E, empty):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(E)
    counts = torch.randint(1, 600, (E,), generator=g)
    if empty == "ends":
        counts[: E // 3] = 0
        counts[E - E // 4:] = 0
    elif empty == "block":
        counts[63:65] = 0
        counts[127:193] = 0
    elif empty == "most":
        counts[torch.rand(E, generator=g) < 0.9] = 0
        counts[E // 2] = 257
    L, K, N = int(counts.sum()), 64, 264
    print(f"persistent experts E={E} {empty} L={L}", flush=True)
    off = counts.cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L, K, generator=g).bfloat16().to(device)
    w = (torch.randn(E, N, K, generator=g) * 0.05).bfloat16().to(device)
    ref = torch.cat([p.float() @ w[e].float().t() for e, p in enumerate(x.split(counts.tolist()))])
    for cfg in (8, 14, 15, 16, 18, 7):  # (16: row tiles of 224, the others of 256 and 160)
        torch.testing.assert_close(ops.scattered_gemm(x, w, 1, ss, off, True, True, cfg=cfg).float(), ref, **TOL)


def test_output_beyond_4_gib(device):
    from dolomite_engine_amd import ops

    counts, K, N = [170001, 0, 100010], 64, 8192
    L = sum(counts)  # 4.4 GB of results; as a pre-activation next to half of that
    print(f"persistent output of {L} x {N}", flush=True)
    g = torch.Generator(device).manual_seed(3)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.empty(L, K, device=device, dtype=torch.bfloat16).normal_(generator=g)
    w = torch.empty(3, N, K, device=device, dtype=torch.bfloat16).normal_(0.0, 0.05, generator=g)
    scattered = ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=8)
    for cfg in (15, 18, 7):
        assert torch.equal(ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=cfg), scattered)
    assert torch.equal(ops.scattered_gemm(x, w.transpose(1, 2).contiguous(), 1, ss, off, True, False, cfg=8, weight_kn=True), scattered)
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    act, h = ops.up_swiglu_keep(by_slot, w, 1, ss, off, cfg=8)
    expert = torch.repeat_interleave(torch.arange(3, device=device), torch.tensor(counts, device=device))
    for rows in torch.arange(L, device=device).split(10000):
        ref = torch.empty(len(rows), N, device=device)
        for e in range(3):
            mine = expert[rows] == e
            ref[mine] = x[rows][mine].float() @ w[e].float().t()
        torch.testing.assert_close(scattered[ss[rows].long()].float(), ref, **TOL)
        torch.testing.assert_close(h[rows].float(), ref, **TOL)
        want = ref[:, :N // 2] * torch.nn.functional.silu(ref[:, N // 2:])
        # (formed from the rounded halves)
        torch.testing.assert_close(act[rows].float(), want, rtol=2.0 ** -6, atol=8e-3)


def test_pre_activation_of_an_expert_beyond_4_gib(device):
    """The pre-activation's rows are addressed from their tile's first, whatever its expert still has behind them: with 262445 rows of
    16 KB in one expert, a tile (of 256 x 256, whose end is the expert's) has just over 4 GiB of them behind its first row."""
    from dolomite_engine_amd import ops

    counts, K, N = [300, 262445], 64, 8192
    L = sum(counts)
    print(f"persistent pre-activation of {L} x {N}", flush=True)
    g = torch.Generator(device).manual_seed(4)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.empty(L, K, device=device, dtype=torch.bfloat16).normal_(generator=g)
    w = torch.empty(2, N, K, device=device, dtype=torch.bfloat16).normal_(0.0, 0.05, generator=g)
    stale = [torch.full((L, n), float("nan"), device=device, dtype=torch.bfloat16) for n in (N, N // 2)]
    del stale  # (what is not written shows: the outputs are allocated where these were)
    act, h = ops.up_swiglu_keep(x, w, 1, ss, off, cfg=8)
    for e, begin, end in ((0, 0, counts[0]), (1, counts[0], L)):
        for rows in torch.arange(begin, end, device=device).split(10000):
            ref = x[ss[rows].long()].float() @ w[e].float().t()
            torch.testing.assert_close(h[rows].float(), ref, **TOL)
            want = ref[:, :N // 2] * torch.nn.functional.silu(ref[:, N // 2:])
            torch.testing.assert_close(act[rows].float(), want, rtol=2.0 ** -6, atol=8e-3)  # (formed from the rounded halves)


def test_pre_activation_rows_of_32_mib(device):
    """Rows of the pre-activation so wide that those of a tile, of 256 or of 160, are beyond 4 GiB."""
    from dolomite_engine_amd import ops

    L, K, N = 300, 8, 2 * ((1 << 23) + 8)
    print(f"pre-activation of {L} x {N}", flush=True)
    g = torch.Generator(device).manual_seed(5)
    off = torch.tensor([L], dtype=torch.int32, device=device)
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.empty(L, K, device=device, dtype=torch.bfloat16).normal_(generator=g)
    w = torch.empty(1, N, K, device=device, dtype=torch.bfloat16).normal_(0.0, 0.05, generator=g)
    stale = [torch.full((L, n), float("nan"), device=device, dtype=torch.bfloat16) for n in (N, N // 2)]
    del stale
    act, h = ops.up_swiglu_keep(x, w, 1, ss, off)
    rows = x[ss.long()].float()
    for cols in torch.arange(N // 2, device=device).split(1 << 18):
        up, gate = rows @ w[0, cols].float().t(), rows @ w[0, N // 2 + cols].float().t()
        torch.testing.assert_close(h[:, cols].float(), up, **TOL)
        torch.testing.assert_close(h[:, N // 2 + cols].float(), gate, **TOL)
        torch.testing.assert_close(act[:, cols].float(), up * torch.nn.functional.silu(gate), rtol=2.0 ** -6, atol=8e-3)
