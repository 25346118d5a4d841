"""The stable expert sort at the sizes where its forms and its chunks change: the four-wave and the sixteen-wave one-block
sort (512 / 513 and 8192 slots, a wave's last step partly filled), more than 963 experts (the one-block sort's counters
beyond 64 KB of LDS), the three passes from 8193 slots on, with a last chunk of one slot, and both sides of the rule that
picks the chunk (by the size of the table and of the workspace).  Integers: exact against numpy's stable sort."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,E", [(1, 1), (63, 5), (512, 40), (513, 40), (1025, 7), (8191, 64), (8192, 1024), (700, 964),
                                 (8193, 17), (8704, 33), (8705, 1000), (8193, 963), (8193, 964), (16383, 1024), (16897, 1024), (300001, 40)])
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


def test_workspace_of_a_larger_batch(device):
    """A workspace sized for 262144 slots serves every smaller batch, in chunks that its table has room for."""
    from dolomite_engine_amd import _lib

    lib = _lib.load()
    E, ws_bytes = 40, lib.mi_moe_sort_bin_workspace_bytes(262144, 40)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=device)
    g = torch.Generator().manual_seed(5)
    for L in (262144, 131072, 65536, 8193):
        ids = torch.randint(0, E, (L,), generator=g, dtype=torch.int32)
        dev_ids = ids.to(device)
        se, ss, off = (torch.empty(n, dtype=torch.int32, device=device) for n in (L, L, E))
        rc = lib.mi_moe_sort_bin(dev_ids.data_ptr(), L, 1, E, se.data_ptr(), ss.data_ptr(), off.data_ptr(), ws.data_ptr(),
                                 ws_bytes, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, L
        assert np.array_equal(ss.cpu().numpy(), np.argsort(ids.numpy(), kind="stable")), L
