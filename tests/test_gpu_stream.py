"""The weight-stream form of the grouped GEMM at the sizes where its units can go wrong: one row, rows around a block of
16 and around a chunk, experts without rows, contractions of one slice, shorter than the ring, with a partial last slice
and of fewer slices than waves, and output columns that end inside a unit.  Against an fp32 product of the same rounded
operands (float64 for fp32): 16-bit results carry one rounding, half a unit in the last place; fp32 results differ by the
order of at most 1000 sums of magnitude below 1 (relative 1e-5 of the largest)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: dict(rtol=2.0 ** -8, atol=2e-3), torch.float16: dict(rtol=2.0 ** -11, atol=5e-4),
       torch.float32: dict(rtol=1e-5, atol=2e-5)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("counts,K,N", [([1], 64, 32), ([0, 1, 0, 17, 16, 15], 136, 72), ([33, 32, 31, 0, 64, 65], 1000, 260),
                                        ([2] * 70, 8, 16), ([5, 0, 3], 512, 1536), ([40, 1], 264, 28)])
@pytest.mark.parametrize("cfg", [-1, 111, 112, 114, 121, 122, 124, 141, 142])
def test_stream_edges(device, dtype, counts, K, N, cfg):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(K + N + len(counts))
    E, L, k = len(counts), sum(counts), 1
    print(f"stream E={E} L={L} K={K} N={N} cfg={cfg} {dtype}", flush=True)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L, K, generator=g).to(dtype).to(device)
    w = (torch.randn(E, 2 * N, K, generator=g) * 0.05).to(dtype).to(device)
    wide = torch.float64 if dtype == torch.float32 else torch.float32
    ref = torch.cat([p.to(wide) @ w[e].to(wide).t() for e, p in enumerate(x.split(counts))])
    plain = ops.scattered_gemm(x, w, k, ss, off, True, False, cfg=cfg)
    torch.testing.assert_close(plain[ss.long()].to(wide), ref, **TOL[dtype])
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    assert torch.equal(ops.scattered_gemm(by_slot, w, k, ss, off, False, False, cfg=cfg), plain)
    act = ops.up_swiglu(by_slot, w, k, ss, off, cfg=cfg)
    want = ref[:, :N] * torch.nn.functional.silu(ref[:, N:])
    torch.testing.assert_close(act.to(wide), want, **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("counts,K,N", [([300, 7, 0, 33], 136, 296), ([16, 17, 129], 1096, 28), ([0, 513], 72, 520)])
@pytest.mark.parametrize("cfg", [-1, 111, 124, 142])
def test_stream_many_chunks(device, dtype, counts, K, N, cfg):
    """Experts of many row chunks beside experts of one: the chunks of a unit are eight blocks apart, in groups of eight units
    of which the last is smaller (10, 1 and 17 units plain; 19, 2 and 33 of SwiGLU).  A row's result does not depend on which
    rows share its chunk: equal to the call in which every expert's rows are in another order, bit for bit."""
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(K + N)
    E, L = len(counts), sum(counts)
    print(f"stream chunks {counts} K={K} N={N} cfg={cfg} {dtype}", flush=True)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L, K, generator=g).to(dtype).to(device)
    w = (torch.randn(E, 2 * N, K, generator=g) * 0.05).to(dtype).to(device)
    wide = torch.float64 if dtype == torch.float32 else torch.float32
    ref = torch.cat([p.to(wide) @ w[e].to(wide).t() for e, p in enumerate(x.split(counts))])
    plain = ops.scattered_gemm(x, w, 1, ss, off, True, True, cfg=cfg)
    torch.testing.assert_close(plain.to(wide), ref, **TOL[dtype])
    other = torch.cat([p.flip(0) for p in torch.arange(L).split(counts)]).to(device)
    assert torch.equal(ops.scattered_gemm(x[other].contiguous(), w, 1, ss, off, True, True, cfg=cfg), plain[other])
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    act = ops.up_swiglu(by_slot, w, 1, ss, off, cfg=cfg)
    want = ref[:, :N] * torch.nn.functional.silu(ref[:, N:])
    torch.testing.assert_close(act.to(wide), want, **TOL[dtype])


@pytest.mark.parametrize("rb,waves", [(1, 1), (1, 4), (2, 2), (4, 1)])
def test_stream_fp32_beyond_one_chunk(device, rb, waves):
    """fp32 beyond one chunk of rows per expert on average is another kernel (no non-temporal fetch for experts with one
    chunk): a row more, past the line, changes no other row's result."""
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(rb)
    K, N, rows, cfg = 520, 296, 32 * rb + 1, 100 + 10 * rb + waves
    print(f"stream fp32 line cfg={cfg}", flush=True)
    x = torch.randn(rows, K, generator=g).to(device)
    w = (torch.randn(2, 2 * N, K, generator=g) * 0.05).to(device)
    out = []
    for first in (rows - 2, rows - 1):  # 16 rb rows per expert on average, and one row more in the first expert
        xs = torch.cat((x[:first], x[-1:]))
        off = torch.tensor([first, first + 1], dtype=torch.int32, device=device)
        ss = torch.arange(first + 1, dtype=torch.int32, device=device)
        out.append((ops.scattered_gemm(xs, w, 1, ss, off, True, True, cfg=cfg), ops.up_swiglu(xs, w, 1, ss, off, cfg=cfg)))
    for at, past in zip(*out):
        assert torch.equal(at[:rows - 2], past[:rows - 2]) and torch.equal(at[-1], past[-1])
