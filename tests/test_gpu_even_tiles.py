"""The even forms of the persistent grouped GEMM: contractions below, at and past the three slices of their ring, with whole and
ragged last slices; experts at the edges of a row tile, of its steps of 32 rows and of four row pairs; columns at the edges of each
tile.  Against an fp32 product of the same rounded operands: one rounding of the result (2^-9 of the value in bf16, 2^-12 in fp16)
plus the order of the fp32 sum; bit for bit against the 256 x 256 tiles, which add in the same order."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: dict(rtol=2.0 ** -8, atol=2e-3), torch.float16: dict(rtol=2.0 ** -11, atol=5e-4)}
ROWS = {14: 256, 15: 160, 16: 224, 18: 256}
COLUMNS = {14: 128, 15: 256, 16: 192, 18: 256}
PLAIN, SWIGLU, KEEP, WEIGHT_KN = range(4)


def _problem(device, counts, K, N, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    E, L = len(counts), sum(counts)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L, K, generator=g).to(dtype).to(device)
    w = (torch.randn(E, N, K, generator=g) * 0.05).to(dtype).to(device)
    ref = torch.cat([p.float() @ w[e].float().t() for e, p in enumerate(x.split(counts))])
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    return off, ss, x, w, ref, by_slot


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [8, 64, 72, 128, 136, 192, 200, 256, 520])
@pytest.mark.parametrize("tile", [14, 15, 16, 18])
def test_even_edges(device, tile, K, dtype):
    from dolomite_engine_amd import ops

    h, n = ROWS[tile], COLUMNS[tile]
    counts = [h, h + 1, 2 * h, 2 * h - 31, 1, 0, 31, 32, 33, 127, 128, 129, 159, 160, 161, 2 * h + 1, 5 * h + 7, 191, 193, 225]
    for N in (n, 2 * n + 16, n - 8 if n % 16 else n - 16):
        print(f"even tile={tile} K={K} N={N} {dtype}", flush=True)
        off, ss, x, w, ref, by_slot = _problem(device, counts, K, N, dtype, K * 7 + N)
        grouped = ops.scattered_gemm(x, w, 1, ss, off, True, True, cfg=tile)
        torch.testing.assert_close(grouped.float(), ref, **TOL[dtype])
        assert torch.equal(grouped, ops.scattered_gemm(x, w, 1, ss, off, True, True, cfg=8))
        assert torch.equal(ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=tile)[ss.long()], grouped)
        assert torch.equal(ops.scattered_gemm(by_slot, w, 1, ss, off, False, True, cfg=tile), grouped)
        act = ops.up_swiglu(by_slot, w, 1, ss, off, cfg=tile)
        want = ref[:, :N // 2] * torch.nn.functional.silu(ref[:, N // 2:])
        torch.testing.assert_close(act.float(), want, **TOL[dtype])
        assert torch.equal(act, ops.up_swiglu(by_slot, w, 1, ss, off, cfg=8))


@pytest.mark.parametrize("tile", [14, 15, 16, 18])
def test_even_many_tiles(device, tile):
    """Several tiles to a workgroup, low and whole ones in turn, and a second block of 64 in its list."""
    from dolomite_engine_amd import ops

    h, n = ROWS[tile], COLUMNS[tile]
    counts = [h, 40, 3 * h, h - 33, 0, 2 * h + 5, 130, 97] * 30
    N = 24 * n - 16
    off, ss, x, w, ref, by_slot = _problem(device, counts, 72, N, torch.bfloat16, tile)
    o = ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=tile)[ss.long()]
    torch.testing.assert_close(o.float(), ref, **TOL[torch.bfloat16])
    act = ops.up_swiglu(by_slot, w, 1, ss, off, cfg=tile)
    torch.testing.assert_close(act.float(), ref[:, :N // 2] * torch.nn.functional.silu(ref[:, N // 2:]), **TOL[torch.bfloat16])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,E,K,N,tile,tile_kn", [(125, 32, 1024, 512, 14, 15), (130, 40, 136, 512, 16, 15), (500, 32, 200, 512, 15, 15),
                                                     (800, 40, 1544, 504, 18, 18), (410, 40, 1536, 512, 15, 15)])
def test_even_training_forms(device, dtype, rows, E, K, N, tile, tile_kn):
    from dolomite_engine_amd import _lib, ops

    counts = [rows] * E
    for e in range(0, E - 1, 2):
        counts[e] -= e % 23
        counts[e + 1] += e % 23
    L = sum(counts)
    off, ss, x, w, ref, by_slot = _problem(device, counts, K, 2 * N, dtype, rows)
    choice = _lib.load().mi_moe_grouped_gemm_tile_choice
    print(f"even training rows={rows} E={E} K={K} N={N}: {choice(L, K, N, E, KEEP)}, {choice(L, K, 2 * N, E, WEIGHT_KN)}", flush=True)
    assert (choice(L, K, N, E, KEEP), choice(L, K, 2 * N, E, WEIGHT_KN)) == (tile, tile_kn)
    plain = ops.scattered_gemm(by_slot, w, 1, ss, off, False, True, cfg=8)
    torch.testing.assert_close(plain.float(), ref, **TOL[dtype])
    want = plain.float()[:, :N] * torch.nn.functional.silu(plain.float()[:, N:])  # (one rounding, and the rounded halves are exact)
    w_kn = w.transpose(1, 2).contiguous()
    for cfg, cfg_kn in ((-1, -1), (tile, tile_kn)):  # by the rule, and the tiles that it names for an even load
        act, h = ops.up_swiglu_keep(by_slot, w, 1, ss, off, cfg=cfg)
        assert torch.equal(h, plain)
        torch.testing.assert_close(act.float(), want, rtol=TOL[dtype]["rtol"], atol=TOL[dtype]["atol"])
        assert torch.equal(ops.scattered_gemm(x, w_kn, 1, ss, off, True, True, cfg=cfg_kn, weight_kn=True), plain)


def test_tile_choice_takes_no_time(device):
    """The rule runs in front of every launch: its time does not grow with the load (1 ms is thirty times less than a sum over all
    row tiles of an expert takes here, and a thousand times what is needed)."""
    import time

    from dolomite_engine_amd import _lib

    choice = _lib.load().mi_moe_grouped_gemm_tile_choice
    times = []
    for _ in range(5):
        start = time.perf_counter()
        choice(1 << 30, 64, 64, 3, PLAIN)
        times.append(time.perf_counter() - start)
    print(f"tile choice of 2^30 rows: {min(times) * 1e6:.1f} us", flush=True)
    assert min(times) < 1e-3


@pytest.mark.parametrize("L,K,N,E", [(1000, 5120, 4096, 8), (2000, 5120, 2048, 8), (2000, 5632, 2048, 8), (4096, 5120, 1024, 16), (1500, 6144, 4096, 8)])
def test_tile_choice_knows_what_is_cut(device, L, K, N, E):
    """Contractions that the persistent kernel may cut along K in principle (5120 on), at loads whose last round it does not cut, as the
    parts would save too little: with a workspace the choice is the same as without one, and not the 256 x 256 tiles.  (One half of the
    chip has one of those: two parts of 40 to 48 slices, of the 60 that they would have to save.)"""
    from dolomite_engine_amd import _lib

    lib = _lib.load()
    assert lib.mi_moe_grouped_gemm_splits(K, 1) == 1
    tile = lib.mi_moe_grouped_gemm_tile_choice(L, K, N, E, PLAIN)
    assert tile != 0
    assert lib.mi_moe_grouped_gemm_tile_choice_ws(L, K, N, E, PLAIN) == tile
