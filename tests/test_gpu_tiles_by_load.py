"""The persistent grouped GEMM that picks its tiles by the experts' rows: every pick, at the ends of its blocks of 64 experts, with
experts that have no rows or nearly all, in all four forms.  Bit for bit against the 256 x 256 tiles, which add in the same order;
where tiles are cut along K, whose parts add in another one, the bits tell which tiles ran."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

PLAIN, SWIGLU, KEEP, WEIGHT_KN = range(4)


def _pick(counts, K, N, form, ws=0):
    from dolomite_engine_amd import _lib

    ends = torch.tensor(counts).cumsum(0).int()
    return _lib.load().mi_moe_grouped_gemm_tile_choice_load(ctypes.c_void_p(ends.data_ptr()), K, N, len(counts), form, ws)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,K,N,picks", [
    ([1], 8, 16, None), ([300, 20], 64, 272, (14, 14, 14, 15)), ([1] * 256, 200, 64, (14, 14, 14, 15)), ([257, 1] * 33, 72, 1040, (15, 15, 15, 15)),
    ([150] * 40, 136, 1040, (16, 16, 16, 15)), ([250] * 65, 200, 528, (0, 0, 0, 0)), ([161, 40, 0, 320] * 10, 64, 1280, (15, 15, 15, 15)),
    ([500] * 32, 72, 1040, (0, 0, 15, 0)), ([700, 10, 0] * 40, 128, 1536, (18, 18, 18, 18)), ([100, 220] * 30, 264, 2064, (16, 16, 16, 18)),
    ([224] * 20, 136, 3088, (14, 14, 14, 18)), ([0] * 63 + [900, 1] + [0] * 63 + [300] * 2 + [0] * 126, 72, 528, None),
    ([0, 0, 5000, 0], 1000, 528, None), ([1000, 2, 0, 1] * 48, 72, 272, None), ([0] * 129 + [4000], 520, 272, None)])
def test_every_pick(device, counts, K, N, picks, dtype):
    from dolomite_engine_amd import ops

    E, L = len(counts), sum(counts)
    got = tuple(_pick(counts, K, N if form in (PLAIN, WEIGHT_KN) else N // 2, form) for form in range(4))
    print(f"by load E={E} L={L} K={K} N={N} {dtype}: {got}", flush=True)
    assert picks is None or torch.cuda.get_device_properties(device).multi_processor_count != 256 or got == picks
    g = torch.Generator().manual_seed(E + L + K)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    x = torch.randn(L, K, generator=g).to(dtype).to(device)
    w = (torch.randn(E, N, K, generator=g) * 0.05).to(dtype).to(device)
    w_kn = w.transpose(1, 2).contiguous()
    for grouped_in, grouped_out in ((True, True), (True, False), (False, True)):
        want = ops.scattered_gemm(x, w, 1, ss, off, grouped_in, grouped_out, cfg=8)
        assert torch.equal(ops.scattered_gemm(x, w, 1, ss, off, grouped_in, grouped_out, cfg=19), want)
        assert torch.equal(ops.scattered_gemm(x, w_kn, 1, ss, off, grouped_in, grouped_out, cfg=19, weight_kn=True), want)
    assert torch.equal(ops.up_swiglu(x, w, 1, ss, off, cfg=19), ops.up_swiglu(x, w, 1, ss, off, cfg=8))
    for a, b in zip(ops.up_swiglu_keep(x, w, 1, ss, off, cfg=19), ops.up_swiglu_keep(x, w, 1, ss, off, cfg=8)):
        assert torch.equal(a, b)


CUT = [([400, 401, 399, 400], 18), ([576, 406, 331, 287], 0), ([10, 20, 30, 1540], 0)]


@pytest.mark.parametrize("counts,pick", CUT)
@pytest.mark.parametrize("form", [PLAIN, SWIGLU, WEIGHT_KN])
def test_load_and_not_average_picks(device, counts, pick, form):
    """Four experts with 400 rows on average, 8192 -> 8192: where they all have about as many, the even tiles are one round; where two
    have more, 256 x 256 tiles whose second round is cut along K.  On average (what the host knows) it is the former."""
    from dolomite_engine_amd import _lib, ops

    if torch.cuda.get_device_properties(device).multi_processor_count != 256:
        pytest.skip("the numbers are those of 256 CUs")
    K = rows = 8192  # weight rows
    N = rows // 2 if form == SWIGLU else rows
    L = sum(counts)
    assert _lib.load().mi_moe_grouped_gemm_tile_choice_ws(L, K, N, 4, form) == 18
    assert _pick(counts, K, N, form, 1) == pick
    print(f"by load with a workspace {counts} form={form}", flush=True)
    g = torch.Generator(device).manual_seed(L)
    off = torch.tensor(counts).cumsum(0).int().to(device)
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.empty(L, K, device=device, dtype=torch.bfloat16).normal_(generator=g)
    w = torch.empty(4, rows, K, device=device, dtype=torch.bfloat16).normal_(0.0, 0.02, generator=g)
    if form == WEIGHT_KN:
        w = w.transpose(1, 2).contiguous()

    def run(cfg):
        if form == SWIGLU:
            return ops.up_swiglu(x, w, 1, ss, off, cfg=cfg)
        return ops.scattered_gemm(x, w, 1, ss, off, True, False, cfg=cfg, weight_kn=form == WEIGHT_KN)

    whole, cut = run(18), run(9)
    assert torch.equal(whole, cut) == (pick == 18)
    for cfg in (7, 19):
        assert torch.equal(run(cfg), whole if pick == 18 else cut)


def test_replays_of_a_graph_follow_the_load(device):
    """The pick is the kernel's: replays of one captured call with other loads in its buffers."""
    from dolomite_engine_amd import ops

    K, N, E, L = 520, 1040, 40, 8000
    g = torch.Generator().manual_seed(9)
    loads = []
    for p in (0.0, 0.3, 0.7, 3.0):
        share = torch.arange(1, E + 1, dtype=torch.float64).pow(-p)[torch.randperm(E, generator=g)]
        loads.append(torch.bincount(torch.multinomial(share, L, replacement=True, generator=g), minlength=E))
    print("by load in a graph", [_pick(c.tolist(), K, N // 2, SWIGLU) for c in loads], flush=True)
    x = torch.randn(L, K, generator=g).bfloat16().to(device)
    w = (torch.randn(E, N, K, generator=g) * 0.05).bfloat16().to(device)
    ss = torch.randperm(L, generator=g).int().to(device)
    off = loads[0].cumsum(0).int().to(device)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops.up_swiglu(x, w, 1, ss, off, cfg=19)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.up_swiglu(x, w, 1, ss, off, cfg=19)
    for _ in range(2):
        for counts in loads:
            off.copy_(counts.cumsum(0).int())
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ops.up_swiglu(x, w, 1, ss, off, cfg=8))
