"""The persistent grouped GEMM at the sizes where its tiles, slices and tile list can go wrong: contractions shorter than
a slice, of exactly one or two slices and with every kind of partial last slice, expert sizes around the 256-row tile,
output columns around the 256- and 128-column tiles, experts without rows, more tiles a workgroup than a block of its tile list
holds (64).  Against an fp32 product of the same rounded operands: fp32 accumulation leaves the one rounding of the
result, half a unit in the last place (2^-9 of the value in bf16, 2^-12 in fp16), plus the reordering error of the fp32
sum, far below the absolute term for these magnitudes."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: dict(rtol=2.0 ** -8, atol=2e-3), torch.float16: dict(rtol=2.0 ** -11, atol=5e-4)}


def _reference(x, w, counts):
    return torch.cat([p.float() @ w[e].float().t() for e, p in enumerate(x.split(counts))])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,K,N", [
    ([300, 20], 8, 264), ([257, 255], 64, 256), ([256, 1], 72, 8), ([511], 120, 136), ([513, 0, 3], 128, 248),
    ([260], 136, 512), ([700, 33], 920, 520), ([1] * 256, 200, 64), ([129, 128, 127], 1000, 1544),
    ([40000], 64, 1024),  # 628 tiles of one expert: several per workgroup
    # so many tiles that the pre-activation form is the persistent kernel's too, with experts that end inside a tile
    ([259, 121, 130] * 13, 72, 1040), ([300, 255, 1, 0, 257, 400] * 8, 64, 1024),
])
def test_persistent_edges(device, dtype, counts, K, N):
    from dolomite_engine_amd import _lib, ops

    g = torch.Generator().manual_seed(K * 7 + N + len(counts))
    E, L = len(counts), sum(counts)
    print(f"persistent E={E} L={L} K={K} N={N} {dtype}", flush=True)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L, K, generator=g).to(dtype).to(device)
    w = (torch.randn(E, N, K, generator=g) * 0.05).to(dtype).to(device)
    ref = _reference(x, w, counts)
    grouped = ops.scattered_gemm(x, w, 1, ss, off, True, True, cfg=8)
    torch.testing.assert_close(grouped.float(), ref, **TOL[dtype])
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    w_kn = w.transpose(1, 2).contiguous()
    half, few = N // 2, True
    if N % 16 == 0:
        want = ref[:, :half] * torch.nn.functional.silu(ref[:, half:])
        keep_tol = dict(rtol=TOL[dtype]["rtol"] * 4, atol=TOL[dtype]["atol"] * 4)
        few = _lib.load().mi_moe_grouped_gemm_choice(L, K, half, E, 1, ops._code(dtype)) != 7
    for cfg in (8, 9, 7):  # the 256 x 256 tiles in both orders, and the tiles that the rule picks
        assert torch.equal(ops.scattered_gemm(x, w, 1, ss, off, True, True, cfg=cfg), grouped)
        scattered = ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=cfg)
        assert torch.equal(scattered[ss.long()], grouped)
        assert torch.equal(ops.scattered_gemm(by_slot, w, 1, ss, off, False, True, cfg=cfg), grouped)
        assert torch.equal(ops.scattered_gemm(x, w_kn, 1, ss, off, True, True, cfg=cfg, weight_kn=True), grouped)
        if N % 16 == 0:
            act = ops.up_swiglu(by_slot, w, 1, ss, off, cfg=cfg)
            torch.testing.assert_close(act.float(), want, **TOL[dtype])
            act_k, h = ops.up_swiglu_keep(by_slot, w, 1, ss, off, cfg=cfg)
            assert torch.equal(h, grouped)
            torch.testing.assert_close(act_k.float(), want, **keep_tol)
    if N % 16 == 0 and L >= 120 * E:
        # (the persistent kernel, or with few tiles the product on smaller ones)
        act_k, h = ops.up_swiglu_keep(by_slot, w, 1, ss, off)
        assert torch.equal(h, ops.scattered_gemm(by_slot, w, 1, ss, off, False, True, cfg=-1 if few else 7))
        torch.testing.assert_close(h.float(), ref, **TOL[dtype])
        torch.testing.assert_close(act_k.float(), want, **keep_tol)


@pytest.mark.parametrize("items,K", [(64, 72), (65, 8), (66, 136), (130, 64)])
@pytest.mark.parametrize("cfg", [8, 9])
def test_persistent_tile_list(device, items, K, cfg):
    """Workgroups with just over one block of their tile list, two and three tiles over, and just over two blocks: 255
    experts of one row and one of 300, of which each XCD or each round has its part."""
    from dolomite_engine_amd import ops

    E, cus = 256, torch.cuda.get_device_properties(device).multi_processor_count
    counts = [1] * 100 + [300] + [1] * 155
    n_tiles = -(-items * cus // (E + 1))  # (257 row tiles)
    assert (E + 1) * n_tiles >= items * cus
    N, L = 256 * n_tiles - 16, sum(counts)
    print(f"persistent tile list items={items} K={K} N={N} cfg={cfg}", flush=True)
    g = torch.Generator(device).manual_seed(items)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.empty(L, K, device=device, dtype=torch.bfloat16).normal_(generator=g)
    w = torch.empty(E, N, K, device=device, dtype=torch.bfloat16).normal_(0.0, 0.05, generator=g)
    ref = _reference(x, w, counts)
    o = ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=cfg)
    torch.testing.assert_close(o[ss.long()].float(), ref, **TOL[torch.bfloat16])
    by_slot = torch.empty_like(x)
    by_slot[ss.long()] = x
    act = ops.up_swiglu(by_slot, w, 1, ss, off, cfg=cfg)
    want = ref[:, :N // 2] * torch.nn.functional.silu(ref[:, N // 2:])
    torch.testing.assert_close(act.float(), want, **TOL[torch.bfloat16])
    w_kn = w.transpose(1, 2).contiguous()
    for form in (cfg, -1):
        assert torch.equal(ops.scattered_gemm(x, w_kn, 1, ss, off, True, False, cfg=form, weight_kn=True), o)
    del w_kn
    act_k, h = ops.up_swiglu_keep(by_slot, w, 1, ss, off, cfg=cfg)
    assert torch.equal(h, o[ss.long()])
    torch.testing.assert_close(act_k.float(), want, rtol=4 * TOL[torch.bfloat16]["rtol"], atol=4 * TOL[torch.bfloat16]["atol"])
