"""The stable expert sort at the sizes where its forms and its chunks change: the four-wave and the sixteen-wave one-block
sort (512 / 513 and 8192 slots, a wave's last step partly filled), more than 963 experts (the one-block sort's counters
beyond 64 KB of LDS), the three passes from 8193 slots on, with a last chunk of one slot, and both sides of the rule that
picks the chunk.  Integers: exact against numpy's stable sort."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,E", [(1, 1), (63, 5), (512, 40), (513, 40), (1025, 7), (8191, 64), (8192, 1024), (700, 964),
                                 (8193, 17), (8704, 33), (8705, 1000), (16383, 1024), (16897, 1024), (300001, 40)])
@pytest.mark.parametrize("skew", [False, True])
def test_sort_edges(device, L, E, skew):
    from dolomite_engine_amd import ops

    g = torch.Generator().manual_seed(L * 3 + E)
    ids = torch.rand(L, generator=g)
    ids = ((ids ** 3 if skew else ids) * E).long().clamp_(max=E - 1).int()
    print(f"sort L={L} E={E} skew={skew}", flush=True)
    se, ss, off = ops.sort_bin(ids.view(L, 1).to(device), E)
    order = np.argsort(ids.numpy(), kind="stable")
    assert np.array_equal(ss.cpu().numpy(), order)
    assert np.array_equal(se.cpu().numpy(), ids.numpy()[order])
    assert np.array_equal(off.cpu().numpy(), np.cumsum(np.bincount(ids.numpy(), minlength=E)))
