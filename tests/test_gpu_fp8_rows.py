"""The persistent fp8 tiles store every tile on one path, in windows of rows that 32-bit offsets reach: experts at the edges of a
tile's blocks of rows, low tiles next to full ones in one workgroup's list, results beyond 4 GiB.
Against an fp32 product of the same operands, tolerance as in test_gpu_fp8_persistent.py: half a unit of the result's last place
(2^-9 of the value in bf16, 2^-12 in fp16) and the reordering error of an fp32 sum, far below the absolute term."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: dict(rtol=2.0 ** -8, atol=2e-3), torch.float16: dict(rtol=2.0 ** -11, atol=5e-4)}
EDGES = [1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 0, 160, 161, 193, 225, 256, 257]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("counts,K,N", [(EDGES, 384, 264), (EDGES, 640, 128), (EDGES[::-1] * 5, 272, 2048), ([257, 1] * 100, 384, 1032)])
def test_row_edges(device, dtype, counts, K, N, tiled):
    from dolomite_engine_amd import ops

    if tiled and K % 128:
        pytest.skip("the streamed-tile layout has whole 128-wide stages")
    print(f"fp8 row edges E={len(counts)} K={K} N={N} tiled={tiled} {dtype}", flush=True)
    g = torch.Generator(device).manual_seed(K + N)
    E, L = len(counts), sum(counts)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.empty(L, K, device=device, dtype=dtype).normal_(generator=g)

    def weights(rows, glu):
        q = torch.empty(E, rows, K, device=device).normal_(0.0, 40.0, generator=g).to(torch.float8_e4m3fn)
        scale = torch.empty(E, rows, device=device).uniform_(5e-4, 1.5e-3, generator=g)
        return (ops.fp8_tile(q, glu) if tiled else q), scale, q.float() * scale.unsqueeze(-1)

    q, scale, wide = weights(2 * N, True)
    h = torch.cat([p @ wide[e].t() for e, p in enumerate(x[ss.long()].float().split(counts))])
    act = ops.up_swiglu_fp8(x, q, scale, 1, ss, off, widen=False, cfg=3)
    torch.testing.assert_close(act.float(), h[:, :N] * torch.nn.functional.silu(h[:, N:]), **TOL[dtype])
    q, scale, wide = weights(N, False)
    o = ops.down_fp8(x, q, scale, ss, off, widen=False, cfg=3)
    want = torch.cat([p @ wide[e].t() for e, p in enumerate(x.float().split(counts))])
    torch.testing.assert_close(o[ss.long()].float(), want, **TOL[dtype])


def test_output_beyond_4_gib(device):
    from dolomite_engine_amd import ops

    counts, K, N, dtype = [170001, 0, 100010], 272, 8192, torch.bfloat16
    L = sum(counts)  # 4.4 GB of results
    print(f"fp8 output of {L} x {N}", flush=True)
    g = torch.Generator(device).manual_seed(5)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.empty(L, K, device=device, dtype=dtype).normal_(generator=g)
    q = torch.empty(3, N, K, device=device).normal_(0.0, 40.0, generator=g).to(torch.float8_e4m3fn)
    scale = torch.empty(3, N, device=device).uniform_(5e-4, 1.5e-3, generator=g)
    o = ops.down_fp8(x, q, scale, ss, off, widen=False, cfg=3)
    for e, begin, end in ((0, 0, 170001), (2, 170001, L)):
        wide = (q[e].float() * scale[e].unsqueeze(-1)).t()
        for rows in torch.arange(begin, end, device=device).split(10000):
            torch.testing.assert_close(o[ss[rows].long()].float(), x[rows].float() @ wide, **TOL[dtype])
