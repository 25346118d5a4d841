"""Grouped GEMMs whose activations end just below, or beyond, the 4 GiB that 32-bit byte offsets reach.  The last rows are
the ones a wrong bound would read as zeros or from the buffer's start."""

import pytest
import torch

from dolomite_engine_amd import ops

pytestmark = pytest.mark.gpu


# bf16: 2^32 - 2080 bytes on the persistent tiles (1032 values a row); fp32: 4 GiB + 4 MiB, few enough results for the
# weight stream, which must leave it to the tiles
@pytest.mark.parametrize("dtype,rows,K,N,tol", [(torch.bfloat16, 2080894, 1032, 8, 2.0**-8), (torch.float32, 262144, 4100, 4, 1e-5)])
def test_last_rows_of_a_4_gib_operand(dtype, rows, K, N, tol):
    x = torch.zeros(rows, K, dtype=dtype, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(3)
    tail = torch.empty(16, K, dtype=dtype, device="cuda").normal_(generator=g)
    x[-16:] = tail
    x[:16] = 3.0
    w = torch.empty(1, N, K, dtype=dtype, device="cuda").normal_(generator=g)
    print(f"operand bytes {dtype} {rows} x {K}", flush=True)
    row_ids = torch.arange(rows, dtype=torch.int32, device="cuda")
    off = torch.full((1,), rows, dtype=torch.int32, device="cuda")
    y = ops.scattered_gemm(x, w, 1, row_ids, off, True, True)
    for got, rows_in in ((y[-16:], tail), (y[:16], x[:16])):
        ref = rows_in.double() @ w[0].double().t()
        # one rounding of the result (bf16), or fp32 sums of K products, against the result's size
        assert (got.double() - ref).norm() <= tol * ref.norm()
    assert (y[16:-16] == 0).all()
