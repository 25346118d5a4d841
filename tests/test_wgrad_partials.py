"""Partial results of the grouped weight gradient: an expert whose rows are cut into groups leaves one fp32 partial result a
group, which a second launch adds up.  They hold the 16 x 16 blocks that exist, not the whole 256 x 256 tiles: a router's
gradient (as many rows as experts, 40 x 1536) is a sixth of its tiles.

The numeric test compares with a product in 64 bits.  Both operands are exact, the sums are fp32 (relative error far below
the rounding of the result for these magnitudes): one rounding, half a unit in the last place (2^-9 of the value in bf16,
2^-12 in fp16), and an absolute term for results that cancel."""

import pytest
import torch


@pytest.mark.parametrize("L,E,M,N", [(32768, 1, 40, 1536), (32768, 1, 8, 4096), (12004, 17, 920, 520), (9000, 7, 136, 1272),
                                     (16384, 1, 64, 4096), (262144, 40, 1024, 1536)])
def test_workspace_holds_blocks_that_exist(L, E, M, N):
    from dolomite_engine_amd import _lib

    got = _lib.load().mi_moe_grouped_wgrad_workspace_bytes(L, E, M, N)
    groups = L // 256 + E  # at most: a group is at least 256 rows, each expert has one that is shorter
    tiles = -(-M // 256) * -(-N // 256)
    chunk = max(256, min(16384, L // -(-384 // tiles)) // 32 * 32)
    if E * tiles >= 256:
        chunk = max(chunk, min(16384, 3 * (L // E) // 2) // 32 * 32)
    blocks = -(-M // 16) * -(-N // 16) * 1024
    plan = 4 * (32 + groups + 3 * E) + 256
    assert got <= (L // chunk + E) * blocks + plan


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,M,N", [
    ([2000], 8, 8), ([3000], 40, 1536), ([2500], 248, 272), ([1030], 264, 136), ([700, 0, 900], 24, 520),
    ([5000, 3, 260], 920, 520), ([257, 256, 4000], 256, 512), ([9000], 136, 1272),
])
def test_partial_results(device, dtype, counts, M, N):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(M * 13 + N)
    L = sum(counts)
    print(f"wgrad partials {counts} {M}x{N} {dtype}", flush=True)
    a = torch.randn(L, M, generator=g).to(dtype).to(device)
    b = torch.randn(L, N, generator=g).to(dtype).to(device)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).to(device)
    want = torch.stack([p.double().t() @ q.double() for p, q in zip(a.split(counts), b.split(counts))])
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    got = ops.grouped_wgrad(a, b, off)
    torch.testing.assert_close(got.double(), want, rtol=eps, atol=2e-3)
    by_slot = torch.empty_like(b)
    by_slot[ss] = b
    assert torch.equal(ops.grouped_wgrad(a, by_slot, off, b_idx=ss.int()), got)
