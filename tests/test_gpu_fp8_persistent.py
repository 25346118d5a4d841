"""The persistent grouped GEMM with fp8 weights at the sizes where its tiles, slices and rings can go wrong: contractions
of exactly three weight slices (the ring's length), with every kind of partial last slice, expert sizes around the
128-row tile and around a wave's 64 rows, output columns that end inside a tile and inside a unit of the streamed-tile
layout, experts without rows, more tiles a workgroup than a block of its tile list holds (64).  Against an fp32 product of the
same operands (e4m3 values are exact in bf16 and fp16): fp32 accumulation leaves the one rounding of the result, half a
unit in the last place (2^-9 of the value in bf16, 2^-12 in fp16), plus the reordering error of the fp32 sum, far below
the absolute term for these magnitudes."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: dict(rtol=2.0 ** -8, atol=2e-3), torch.float16: dict(rtol=2.0 ** -11, atol=5e-4)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,K,N,k", [
    ([1], 272, 8, 1), ([127, 129], 288, 264, 1), ([128, 0, 64], 384, 128, 2), ([65, 63, 0, 1], 400, 136, 3),
    ([300, 20], 512, 1408, 4), ([16] * 8, 1408, 520, 2), ([1] * 255 + [129], 336, 64, 1), ([513, 5, 250], 1024, 256, 6),
    ([9000], 384, 2048, 1),  # 71 row tiles x 16 column tiles
    ([40000, 2], 272, 4096, 2),
])
@pytest.mark.parametrize("tiled", [False, True])
def test_fp8_persistent_edges(device, dtype, counts, K, N, k, tiled):
    from dolomite_engine_amd import ops

    if tiled and K % 128:
        pytest.skip("the streamed-tile layout has whole 128-wide stages")
    g = torch.Generator().manual_seed(K * 7 + N + len(counts))
    E, L = len(counts), sum(counts)
    k = k if L % k == 0 else 1
    print(f"fp8 persistent E={E} L={L} K={K} N={N} k={k} tiled={tiled} {dtype}", flush=True)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L // k, K, generator=g).to(dtype).to(device)

    def weights(rows, glu):
        q = (torch.randn(E, rows, K, generator=g) * 40).to(torch.float8_e4m3fn).to(device)
        scale = (torch.rand(E, rows, generator=g) * 1e-3 + 5e-4).to(device)
        wide = q.float() * scale.unsqueeze(-1)
        return (ops.fp8_tile(q, glu) if tiled else q), scale, wide

    by_row = x.float()[(ss // k).long()]
    q, scale, wide = weights(2 * N, True)
    h = torch.cat([p @ wide[e].t() for e, p in enumerate(by_row.split(counts))])
    act = ops.up_swiglu_fp8(x, q, scale, k, ss, off, widen=False, cfg=3)
    want = h[:, :N] * torch.nn.functional.silu(h[:, N:])
    torch.testing.assert_close(act.float(), want, **TOL[dtype])
    q, scale, wide = weights(N, False)
    rows = by_row.to(dtype)
    o = ops.down_fp8(rows, q, scale, ss, off, widen=False, cfg=3)
    want = torch.cat([p @ wide[e].t() for e, p in enumerate(rows.float().split(counts))])
    torch.testing.assert_close(o[ss.long()].float(), want, **TOL[dtype])


@pytest.mark.parametrize("items,K", [(64, 272), (65, 288), (66, 400), (130, 272)])
def test_fp8_persistent_tile_list(device, items, K):
    """Workgroups with just over one block of their tile list, two and three tiles over, and just over two blocks: 255
    experts of one row and one of 150."""
    from dolomite_engine_amd import ops

    E, cus, dtype = 256, torch.cuda.get_device_properties(device).multi_processor_count, torch.bfloat16
    counts = [1] * 100 + [150] + [1] * 155
    n_tiles = -(-items * cus // (E + 1))  # (257 row tiles)
    N, L = 256 * n_tiles - 16, sum(counts)
    print(f"fp8 persistent tile list items={items} K={K} N={N}", flush=True)
    g = torch.Generator(device).manual_seed(items)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.empty(L, K, device=device, dtype=dtype).normal_(generator=g)
    q = torch.empty(E, N, K, device=device, dtype=dtype).normal_(0.0, 40.0, generator=g).to(torch.float8_e4m3fn)
    scale = torch.empty(E, N, device=device).uniform_(5e-4, 1.5e-3, generator=g)
    ref = torch.cat([p.float() @ (q[e].float() * scale[e].unsqueeze(-1)).t() for e, p in enumerate(x.split(counts))])
    o = ops.down_fp8(x, q, scale, ss, off, widen=False, cfg=3)
    torch.testing.assert_close(o[ss.long()].float(), ref, **TOL[dtype])
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    act = ops.up_swiglu_fp8(by_slot, q, scale, 1, ss, off, widen=False, cfg=3)
    want = ref[:, :N // 2] * torch.nn.functional.silu(ref[:, N // 2:])
    torch.testing.assert_close(act.float(), want, **TOL[dtype])
