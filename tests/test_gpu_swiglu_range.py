"""SwiGLU over the whole range of its operands, in every kernel that has it in its epilogue: up * silu(gate) is finite
wherever silu(gate) times up is, also where up * gate overflows fp32 (bf16 reaches 3e38), and infinities and NaN come out
as torch's ``up * silu(gate)`` gives them.  And the error of the fp8 tiles against 64-bit products: the persistent ones add the
contraction in another order than the register-staged ones, which must not cost accuracy."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# (up, gate): overflowing products with finite results, both signs; the exponential's overflow; infinities and NaN
PAIRS = [(1e20, -1e20), (-1e20, -1e20), (3e38, -200.0), (-1e30, -1e30), (1e25, -100.0), (2.0, 1e30), (1e10, 1e10), (0.0, -3e38),
         (1.0, float("inf")), (float("inf"), 2.0), (0.5, float("nan")), (3.0, -5.0), (-7.0, 0.25), (1e38, 1e-30), (1e-30, -80.0)]


def _torch_swiglu(up, gate):
    return up * torch.nn.functional.silu(gate)


def _operands(device, dtype):
    """Rows whose up / gate results are the pairs: two contraction values, each with a weight of one on its own side."""
    pairs = [p for p in PAIRS if dtype == torch.bfloat16 or all(abs(v) < 6e4 or v != v or v in (float("inf"),) for v in p)]
    up = torch.tensor([p[0] for p in pairs], device=device).to(dtype)
    gate = torch.tensor([p[1] for p in pairs], device=device).to(dtype)
    return up, gate


def _check(act, up, gate, dtype):
    want = _torch_swiglu(up.float(), gate.float())
    # one rounding of the result on top of a few units in the last place of fp32 (exponential, reciprocal)
    rtol = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for n in range(act.shape[1]):
        torch.testing.assert_close(act[:, n].float(), want.to(dtype).float(), rtol=rtol, atol=1e-30, equal_nan=True)


@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4, 5, 7, 111, 122, 141])
def test_swiglu_of_large_operands(device, cfg):
    from dolomite_engine_amd import ops

    dtype = torch.bfloat16
    up, gate = _operands(device, dtype)
    L, K, N = up.numel(), 64, 16
    # (an infinite or NaN operand times the other side's zero weight would be NaN everywhere: each such value has rows of
    # its own below; here the finite pairs)
    finite = torch.isfinite(up) & torch.isfinite(gate)
    up, gate = up[finite], gate[finite]
    L = up.numel()
    x = torch.zeros(L, K, dtype=dtype, device=device)
    x[:, 0], x[:, 1] = up, gate
    w = torch.zeros(1, 2 * N, K, dtype=dtype, device=device)
    w[0, :N, 0] = 1
    w[0, N:, 1] = 1
    ss = torch.arange(L, dtype=torch.int32, device=device)
    off = torch.full((1,), L, dtype=torch.int32, device=device)
    print(f"swiglu range cfg={cfg}", flush=True)
    _check(ops.up_swiglu(x, w, 1, ss, off, cfg=cfg), up, gate, dtype)


def test_swiglu_keep_of_large_operands(device):
    from dolomite_engine_amd import ops

    dtype = torch.bfloat16
    up, gate = _operands(device, dtype)
    finite = torch.isfinite(up) & torch.isfinite(gate)
    up, gate = up[finite].repeat(40), gate[finite].repeat(40)
    L, K, N = up.numel(), 64, 16
    x = torch.zeros(L, K, dtype=dtype, device=device)
    x[:, 0], x[:, 1] = up, gate
    w = torch.zeros(1, 2 * N, K, dtype=dtype, device=device)
    w[0, :N, 0] = 1
    w[0, N:, 1] = 1
    ss = torch.arange(L, dtype=torch.int32, device=device)
    off = torch.full((1,), L, dtype=torch.int32, device=device)
    for cfg in (-1, 8, 14, 15, 16, 18):  # (so few tiles are two launches by themselves)
        act, h = ops.up_swiglu_keep(x, w, 1, ss, off, cfg=cfg)
        assert torch.equal(h[:, 0], up) and torch.equal(h[:, N], gate)
        _check(act, up, gate, dtype)
        _check(ops.swiglu_forward(h), up, gate, dtype)


@pytest.mark.parametrize("cfg", [7, 8, 1, 111])
def test_swiglu_split_and_non_finite(device, cfg):
    """Infinities and NaN come through the gate's own product: a row's only non-zero value is the gate's, and up is a sum of
    the same value (up == gate), so that no zero weight meets an infinity."""
    from dolomite_engine_amd import ops

    dtype = torch.bfloat16
    v = torch.tensor([float("inf"), float("nan"), -1e30, 1e30, -90.0, 2.0], device=device).to(dtype)
    L, K, N = v.numel(), 64, 16
    x = v[:, None].expand(L, K).contiguous()
    w = torch.full((1, 2 * N, K), 1.0 / K, dtype=dtype, device=device)
    ss = torch.arange(L, dtype=torch.int32, device=device)
    off = torch.full((1,), L, dtype=torch.int32, device=device)
    _check(ops.up_swiglu(x, w, 1, ss, off, cfg=cfg), v, v, dtype)


def test_swiglu_of_large_operands_split_k(device):
    """The launch that adds the parts of tiles cut along the contraction has a SwiGLU of its own."""
    from dolomite_engine_amd import ops

    dtype = torch.bfloat16
    up, gate = _operands(device, dtype)
    finite = torch.isfinite(up) & torch.isfinite(gate)
    # 256 rows: one row tile of the two that the launch has to allow for, so every tile is cut in two
    up, gate = up[finite].repeat(22)[:256], gate[finite].repeat(22)[:256]
    L, K, N = up.numel(), 8192, 4096
    x = torch.zeros(L, K, dtype=dtype, device=device)
    x[:, 0], x[:, 1] = up, gate
    w = torch.zeros(1, 2 * N, K, dtype=dtype, device=device)
    w[0, :N, 0] = 1
    w[0, N:, 1] = 1
    ss = torch.arange(L, dtype=torch.int32, device=device)
    off = torch.full((1,), L, dtype=torch.int32, device=device)
    act = ops.up_swiglu(x, w, 1, ss, off, cfg=9)
    assert torch.equal(act, ops.up_swiglu(x, w, 1, ss, off, cfg=9, split_k=False))
    _check(act[:, ::509], up, gate, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cfg", [0, 3, 4])
def test_swiglu_of_large_operands_fp8(device, dtype, cfg):
    from dolomite_engine_amd import ops

    up, gate = _operands(device, torch.bfloat16)
    finite = torch.isfinite(up) & torch.isfinite(gate)
    up, gate = up[finite], gate[finite]
    if dtype == torch.float16:  # the scales supply the range that fp16 activations do not have; results are fp16
        up = torch.tensor([6e4, -6e4, 5e4, -2.0, 3.0], device=device)
        gate = torch.tensor([-6e4, -6e4, -5e4, 0.5, -4.0], device=device)
    L, K, N = up.numel(), 384, 16
    s = 1.0 if dtype == torch.bfloat16 else 2.0 ** 56
    x = torch.zeros(L, K, dtype=dtype, device=device)
    x[:, 0], x[:, 1] = up.to(dtype), gate.to(dtype)
    up, gate = x[:, 0].float(), x[:, 1].float() * s
    if dtype == torch.float16:
        up = up * s
        keep = gate < -1e20  # (the others overflow fp16's results)
        x, up, gate = x[keep].contiguous(), up[keep], gate[keep]
        L = up.numel()
    q = torch.zeros(1, 2 * N, K, device=device)
    q[0, :N, 0] = 1
    q[0, N:, 1] = 1
    scale = torch.full((1, 2 * N), s, device=device)
    ss = torch.arange(L, dtype=torch.int32, device=device)
    off = torch.full((1,), L, dtype=torch.int32, device=device)
    print(f"swiglu range fp8 cfg={cfg} {dtype}", flush=True)
    act = ops.up_swiglu_fp8(x, q.to(torch.float8_e4m3fn), scale, 1, ss, off, widen=False, cfg=cfg)
    _check(act, up, gate, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("E,rows,H,I", [(4, 24, 4096, 1408), (4, 96, 4096, 1408), (3, 200, 1536, 512), (2, 400, 1000, 520)])
def test_fp8_tiles_error_against_64_bits(device, dtype, E, rows, H, I):
    """Both forms of the tiles are one rounding of an fp32 sum away from the 64-bit result; the persistent form's error is
    within 2 % of the staged form's (the two round differently where a sum falls close to the middle of two 16-bit values:
    with n >= 5e4 results the relative errors' norms agree to about n^-1/2, 0.5 %)."""
    from dolomite_engine_amd import ops

    if H % 16:
        H += 16 - H % 16
    g = torch.Generator(device="cuda").manual_seed(E * rows + H)
    L = E * rows
    off = torch.arange(1, E + 1, device=device, dtype=torch.int32) * rows
    ss = torch.randperm(L, generator=g, device=device).int()
    x = torch.randn(L, H, generator=g, device=device).to(dtype)
    w = torch.randn(E, 2 * I, H, generator=g, device=device) * 0.02
    scale = w.abs().amax(-1).clamp_min(1e-12) / 448
    q = (w / scale.unsqueeze(-1)).to(torch.float8_e4m3fn)
    wide = q.double() * scale.double().unsqueeze(-1)
    rows_in = x.double()[ss.long()].view(E, rows, H)
    h = torch.stack([rows_in[e] @ wide[e].t().contiguous() for e in range(E)])
    want = (h[..., :I] * torch.nn.functional.silu(h[..., I:])).view(L, I)

    def error(got):
        return ((got.double() - want).norm() / want.norm()).item()

    errs = [error(ops.up_swiglu_fp8(x, q, scale, 1, ss, off, widen=False, cfg=cfg)) for cfg in (4, 3)]
    print(f"fp8 up-projection {E} x {rows}, {H} -> {I} {dtype}: staged {errs[0]:.4e}, persistent {errs[1]:.4e}", flush=True)
    # one rounding: uniform within half a unit in the last place, at most 2^-9 / 2^-12 of the value
    assert errs[1] <= 1.02 * errs[0] and errs[1] < (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12)
