"""Weight gradients of few rows per expert, which run without a plan: whole experts, one item a tile.  The sizes sit on both sides of
the lines that choose (640 rows of one expert, 768 rows per expert on average, as many as one expert can have), with experts that
have no rows, fewer than a slice of 64, and whole slices.

Against a product in 64 bits: operands are exact, the sums are fp32 (relative error far below the rounding of the result), one
rounding of at most 2^-8 (bf16, 8 significant bits) or 2^-11 (fp16, 11) of the value, and an absolute term for results that cancel: fp32 partial sums
err by at most rows * 2^-24 of the sum of the magnitudes, which is below 0.64 rows for products of two unit normals."""

import os
import re
import shutil
import subprocess

import pytest
import torch

from test_built_kernels import _early_uses, _foreign, _objdump


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gather", ["none", "a", "b"])
@pytest.mark.parametrize("counts,M,N", [
    ([1], 8, 8), ([640], 32, 1024), ([641], 40, 264), ([0, 0, 5], 264, 24), ([64, 0, 63, 65, 128, 0, 300], 520, 248),
    ([1535, 1], 136, 520), ([1535, 2], 136, 520), ([127] * 30 + [0, 2], 264, 264), ([0, 0], 256, 256),
])
def test_whole_experts(device, dtype, gather, counts, M, N):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(M * 17 + N + len(counts))
    L, E = sum(counts), len(counts)
    print(f"wgrad whole {counts[:8]} {M}x{N} {dtype} {gather}", flush=True)
    rows = max(L, 1)
    a, b = torch.randn(rows, M, generator=g).to(dtype), torch.randn(rows, N, generator=g).to(dtype)
    idx = torch.randint(0, rows, (L,), generator=g)
    ai = idx if gather == "a" else torch.arange(L)
    bi = idx if gather == "b" else torch.arange(L)
    off = torch.tensor(counts).cumsum(0)
    want = torch.zeros(E, M, N, dtype=torch.float64)
    for e, n in enumerate(counts):
        r = slice(int(off[e]) - n, int(off[e]))
        want[e] = a[ai[r]].double().t() @ b[bi[r]].double()
    dev = lambda t: t.to(torch.int32).to(device)
    got = ops.grouped_wgrad(a[:L].to(device) if gather != "a" else a.to(device), b[:L].to(device) if gather != "b" else b.to(device),
                            dev(off), dev(idx) if gather == "a" else None, dev(idx) if gather == "b" else None)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = eps * want.abs() + max(counts) * 0.64 * max(counts) * 2.0 ** -24 + 2.0 ** -24
    assert ((got.cpu().double() - want).abs() <= bound).all()


# (tokens, experts, top-k, M, N) at both sides of the bound on what one expert can have: 1024 + 32 rows for each of the k experts' tiles
HOT = [(1088, 3, 1, 264, 8, 1), (1089, 3, 1, 264, 8, 0), (1409, 8, 2, 520, 264, 0), (1408, 8, 2, 520, 264, 1),
       (2048, 40, 2, 1024, 1024, 1), (2049, 40, 2, 1024, 1024, 0), (3073, 40, 8, 1024, 512, 0), (3072, 40, 8, 1024, 512, 1), (32768, 64, 1, 1024, 1024, 0), (6000, 8, 1, 4096, 4096, 1),
       (768, 2, 1, 8, 8, 1), (1057, 2, 1, 8, 8, 0)]


@pytest.mark.parametrize("T,E,k,M,N,whole", HOT)
def test_choice(T, E, k, M, N, whole):
    from dolomite_engine_amd import _lib

    choose = _lib.load().mi_moe_grouped_wgrad_whole
    assert choose(T * k, T * k, T, M, N, E) == choose(T * k, T, T * k, M, N, E) == whole


def test_choice_by_the_average():
    from dolomite_engine_amd import _lib

    choose = _lib.load().mi_moe_grouped_wgrad_whole
    assert choose(640, 640, 640, 32, 1024, 1) == 1 and choose(641, 641, 641, 32, 1024, 1) == 0
    assert choose(6144, 6144, 768, 256, 256, 8) == 1 and choose(6152, 6152, 769, 256, 256, 8) == 0
    assert choose(32768, 32768, 4096, 4096, 4096, 64) == 1 and choose(32776, 32776, 4097, 4096, 4096, 64) == 0
    assert choose(0, 0, 0, 8, 8, 4) == 1 and choose(-1, 0, 0, 8, 8, 1) < 0


@pytest.mark.parametrize("T,H,E,k,I,whole", [(509, 1024, 32, 8, 512, True), (1000, 4096, 8, 2, 14336, True), (640, 64, 8, 1, 8, True),
                                             (4097, 256, 8, 2, 520, False)])
def test_training_call_has_no_room_for_partial_results_that_whole_experts_do_not_leave(T, H, E, k, I, whole):
    import ctypes

    from dolomite_engine_amd import _lib

    lib = _lib.load()
    sizes = [ctypes.c_size_t() for _ in range(3)]
    assert lib.mi_moe_layer_train_sizes(T, H, E, k, I, 2, *(ctypes.byref(s) for s in sizes)) == 0
    L = T * k
    # gradient of the activation with the gated activation, or the slots' gradient of x; d h, d gates, tokens, d logits, the router's d x
    operands = [max(4 * L * I, 2 * L * H), 4 * L * I, 2 * L, 4 * L, 2 * T * E, 2 * T * H]
    # (the gate's gradient is one expert's: its partial results are counted from 641 rows on)
    gate = 0 if T <= 640 else lib.mi_moe_grouped_wgrad_workspace_bytes(T, 1, E, H)
    most = sum(operands) + max(0, gate - operands[0]) + 512 * len(operands)
    slabs = lib.mi_moe_grouped_wgrad_workspace_bytes(L, E, 2 * I, H)
    assert sizes[2].value <= most if whole else sizes[2].value >= slabs


@pytest.mark.gpu
@pytest.mark.parametrize("load", ["even", "hot"])
@pytest.mark.parametrize("T,E,k,M,N,whole", [h for h in HOT if h[0] * h[2] * h[3] * h[4] < 1 << 32])
def test_gathered_by_token(device, load, T, E, k, M, N, whole):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(T + M)
    score = torch.rand(T, E, generator=g)
    if load == "hot":
        score[:, E - k:] += 1  # every token chooses the same experts
    sel, ss = score.topk(k, dim=1).indices.flatten().sort(stable=True)
    off, tok = torch.bincount(sel, minlength=E).cumsum(0), ss // k
    print(f"wgrad by token T={T} E={E} k={k} {M}x{N} {load}", flush=True)
    a, b = torch.randn(T * k, M, generator=g).bfloat16().to(device), torch.randn(T, N, generator=g).bfloat16().to(device)
    got = ops.grouped_wgrad(a, b, off.int().to(device), None, tok.int().to(device))
    turned = ops.grouped_wgrad(b, a, off.int().to(device), tok.int().to(device), None)
    rows = torch.bincount(sel, minlength=E).tolist()
    want = torch.stack([p.double().t() @ q.double() for p, q in zip(a.split(rows), b[tok.to(device)].split(rows))])
    bound = 2.0 ** -8 * want.abs() + max(rows) * 0.64 * max(rows) * 2.0 ** -24 + 2.0 ** -24
    assert ((got.double() - want).abs() <= bound).all()
    assert ((turned.transpose(1, 2).double() - want).abs() <= bound).all()


def test_built_code(tmp_path):
    """The accumulators and row indices of these kernels are used as test_built_kernels.py says of the planned ones."""
    from dolomite_engine_amd import _lib, build, is_built

    if not is_built():
        build()
    shutil.copy(os.path.realpath(_lib.load()._name), tmp_path / "lib.so")
    subprocess.run([_objdump(), "--offloading", str(tmp_path / "lib.so")], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    found = 0
    for image in sorted(p for p in tmp_path.iterdir() if "gfx950" in p.name):
        text = subprocess.run([_objdump(), "-d", "--no-show-raw-insn", "--no-leading-addr", str(image)], check=True,
                              capture_output=True, text=True).stdout
        for label, body in re.findall(r"^(?:[0-9a-f]+ )?<(\w+)>:\n((?:(?!^(?:[0-9a-f]+ )?<).*\n?)*)", text, re.M):
            if "grouped_wgrad_whole_kernelI" not in label:
                continue
            found += 1
            code = [line.split("//")[0].strip() for line in body.splitlines()]
            assert sum("v_mfma" in i for i in code) >= 128
            assert _foreign(code) == [] and _early_uses(code) == []
    assert found == 8
