"""128 x 128 tiles that come by DMA with a contraction that is no multiple of 32 (at most one to a CU), at its edges: 8, 16 and 24 values
in the last slice, fewer slices than the ring has stages, ragged rows and columns, the largest number of tiles and one more.

Against an fp32 product of the same rounded operands: one rounding of the result (2^-8 of the value in bf16, 2^-11 in fp16), plus the
reordering error of the fp32 sum."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: dict(rtol=2.0 ** -8, atol=2e-3), torch.float16: dict(rtol=2.0 ** -11, atol=5e-4)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,K,N", [([5], 8, 4), ([130, 0, 1], 24, 132), ([127, 129], 40, 64), ([300], 104, 260), ([64] * 9, 136, 12),
                                        ([3001], 920, 344), ([128] * 16, 472, 1024), ([128] * 17, 472, 1024)])
def test_ragged_contraction(device, dtype, counts, K, N):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(K + N)
    E, L = len(counts), sum(counts)
    print(f"dma ragged {counts[:4]} K={K} N={N} {dtype}", flush=True)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L, K, generator=g).to(dtype).to(device)
    w = (torch.randn(E, 2 * N, K, generator=g) * 0.05).to(dtype).to(device)
    ref = torch.cat([p.float() @ w[e].float().t() for e, p in enumerate(x.split(counts))])
    torch.testing.assert_close(ops.scattered_gemm(x, w, 1, ss, off, True, True, cfg=1).float(), ref, **TOL[dtype])
    torch.testing.assert_close(ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=1)[ss.long()].float(), ref, **TOL[dtype])
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    up = ops.up_swiglu(by_slot, w, 1, ss, off, cfg=1)
    torch.testing.assert_close(up.float(), ref[:, :N] * torch.nn.functional.silu(ref[:, N:]), **TOL[dtype])


def test_a_rows_neighbours_stay_out(device):
    """What lies behind a row's end is the next row's, and may be infinite."""
    from dolomite_engine_amd import ops

    K, N, L = 40, 24, 40
    x, w = torch.randn(L, K, device=device).bfloat16(), torch.randn(1, N, K, device=device).bfloat16()
    x[1::2] = float("inf")
    w[:, 1::2] = float("nan")
    off, ss = torch.tensor([L], device=device).int(), torch.arange(L, device=device).int()
    out = ops.scattered_gemm(x, w, 1, ss, off, True, True, cfg=1)
    want = x[::2].float() @ w[0, ::2].float().t()
    torch.testing.assert_close(out[::2, ::2].float(), want, **TOL[torch.bfloat16])
