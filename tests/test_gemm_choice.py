"""Which kernel the grouped GEMM picks, at both sides of the lines of its rule (mi_moe_grouped_gemm_choice; host code only).  Numbers as in include/mi_moe.h: 100 + 10 x row blocks + waves is the weight stream, 7 the persistent
256 x 256 tiles, 4 and 1 the 128 x 128 tiles with and without DMA, 5 and 2 the 32-row tiles, 0 the register-staged 256 x 256."""

import pytest

F32, F16, BF16 = 0, 1, 2


def choice(L, K, N, E, glu, dtype=BF16):
    from dolomite_engine_amd import _lib

    return _lib.load().mi_moe_grouped_gemm_choice(L, K, N, E, glu, dtype)


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("at,past,K,N,E,glu", [
    # the weight stream: 16 rows per expert, 24 from K 1280 on, below 48 from K 4096 on, 56 where K is ragged
    ((128, 114), (129, 4), 1024, 512, 8, 0), ((128, 114), (129, 5), 1248, 512, 8, 1), ((192, 124), (193, 5), 1280, 512, 8, 1),
    ((383, 142), (384, 4), 4096, 512, 8, 1), ((448, 141), (449, 1), 920, 520, 8, 1),
    # its forms: 13 rows per expert for long contractions, 16 else, 28; waves by units and slices
    ((520, 112), (521, 122), 1536, 512, 40, 0), ((640, 112), (641, 122), 200, 512, 40, 0), ((1120, 122), (1121, 141), 200, 512, 40, 0),
    ((10, 114), (11, 112), 1536, 512, 40, 1), ((20, 112), (21, 111), 1536, 512, 40, 1), ((64, 114), (65, 111), 4096, 512, 80, 1),
    # 48 rows per expert: the 32 x 128 tiles; below them only short and long contractions take the DMA tiles
    ((1919, 5), (1920, 4), 1536, 512, 40, 1), ((1919, 4), (1919, 5), (1024, 1056), 512, 40, 1),
    # 120 rows per expert: the persistent tiles
    ((4799, 4), (4800, 7), 1536, 512, 40, 1),
    # ... unless there are at most 72 of them, or at most one 128 x 128 tile to a CU with a quarter to spare
    ((4608, 4), (4609, 7), 256, 1024, 1, 0), ((2125, 4), (2250, 7), 512, 768, (17, 18), 1),
    # ... or, with a ragged contraction, at most two to a CU
    ((4000, 1), (4125, 7), 200, 1024, (32, 33), 1),
    # results that the persistent tiles do not take
    ((8176, 1), (8192, 0), 520, 1028, 16, 0),
])
def test_lines(dtype, at, past, K, N, E, glu):
    Ks, Es = (K if isinstance(K, tuple) else (K, K)), (E if isinstance(E, tuple) else (E, E))
    for (L, want), k, e in zip((at, past), Ks, Es):
        assert choice(L, k, N, e, glu, dtype) == want, (L, k, N, e)


@pytest.mark.parametrize("L,K,N,E,glu,want", [
    (128, 256, 512, 8, 1, 114), (512, 256, 512, 8, 1, 111), (2048, 256, 512, 8, 1, 111), (2049, 256, 512, 8, 1, 2),
    (65536, 1536, 512, 8, 1, 1), (2560, 1000, 512, 40, 0, 111), (2561, 1000, 512, 40, 0, 2), (100, 1000, 520, 17, 0, 114),
])
def test_fp32(L, K, N, E, glu, want):
    assert choice(L, K, N, E, glu, F32) == want


def test_refusals():
    from dolomite_engine_amd import _lib

    assert choice(100, 12, 8, 1, 0) == _lib.MI_MOE_EUNSUPPORTED
    assert choice(100, 16, 6, 1, 0) == _lib.MI_MOE_EUNSUPPORTED
    assert choice(100, 12, 8, 1, 0, F32) >= 0
    assert choice(0, 16, 8, 1, 0) == -2 and choice(100, 16, 8, 0, 0) == -2 and choice(100, 16, 8, 1, 0, 7) == -3
