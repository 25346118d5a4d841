"""The grouped GEMM's choice of a kernel by rows per expert and number of tiles, at both sides of its lines: 48 and 120 rows
per expert, 72 and 73 or more 256 x 256 tiles, a 128 x 128 tile or more to a CU, contractions that are and are not multiples of
32, one expert without index arrays' order.  The kernel that runs is the one the rule names (tests/test_gemm_choice.py: which
that is): its result is that configuration's, bit for bit.  Against an fp32 product of the same rounded operands: one rounding of
the result, half a unit in the last place (2^-9 of the value in bf16, 2^-12 in fp16), plus the reordering error of the fp32
sum."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: dict(rtol=2.0 ** -8, atol=2e-3), torch.float16: dict(rtol=2.0 ** -11, atol=5e-4)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("E,rows,K,N", [(4, 47, 1536, 264), (4, 48, 1536, 264), (24, 119, 512, 512), (24, 120, 512, 512),
                                        (24, 129, 520, 520), (1, 3001, 920, 344), (1, 4608, 256, 512), (1, 4609, 256, 512),
                                        (1, 120, 64, 24), (36, 250, 200, 256), (37, 250, 200, 256),
                                        (40, 119, 512, 512), (40, 120, 512, 512), (17, 125, 256, 768), (18, 125, 256, 768),
                                        (32, 125, 200, 1024), (33, 125, 200, 1024), (40, 13, 512, 256), (40, 17, 520, 256),
                                        (40, 57, 520, 256), (16, 512, 520, 1028)])
def test_tile_choice(device, dtype, E, rows, K, N):
    from dolomite_engine_amd import _lib, ops

    g = torch.Generator().manual_seed(E * 1000 + rows)
    counts = [rows] * E
    for e in range(0, E - 1, 2):  # uneven around the average
        d = int(torch.randint(0, rows // 3 + 1, (1,), generator=g))
        counts[e] -= d
        counts[e + 1] += d
    L = sum(counts)
    print(f"tile choice E={E} rows={rows} K={K} N={N} {dtype}", flush=True)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L, K, generator=g).to(dtype).to(device)
    w = (torch.randn(E, 2 * N, K, generator=g) * 0.05).to(dtype).to(device)
    ref = torch.cat([p.float() @ w[e].float().t() for e, p in enumerate(x.split(counts))])
    o = ops.scattered_gemm(x, w, 1, ss, off, True, False)
    torch.testing.assert_close(o[ss.long()].float(), ref, **TOL[dtype])
    named = [_lib.load().mi_moe_grouped_gemm_choice(L, K, n, E, glu, ops._code(dtype)) for n, glu in ((2 * N, 0), (N, 1))]
    print(f"  configurations {named}", flush=True)
    assert torch.equal(ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=named[0], split_k=False), o)
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    want = ref[:, :N] * torch.nn.functional.silu(ref[:, N:])
    up = ops.up_swiglu(by_slot, w, 1, ss, off)
    torch.testing.assert_close(up.float(), want, **TOL[dtype])
    assert torch.equal(ops.up_swiglu(by_slot, w, 1, ss, off, cfg=named[1]), up)
    act, h = ops.up_swiglu_keep(by_slot, w, 1, ss, off)
    torch.testing.assert_close(h.float(), ref, **TOL[dtype])
    # (formed from the rounded halves: two more roundings of a factor each, and silu's slope)
    torch.testing.assert_close(act.float(), want, rtol=TOL[dtype]["rtol"] * 4, atol=TOL[dtype]["atol"] * 4)
