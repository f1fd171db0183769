"""The persistent forward's items where workgroups have one or two at most (host function shared with
the device code)."""
import numpy as np
import pytest

import metalllm_amd as M


@pytest.mark.parametrize("B,T,H,grid", [(1, 8192, 12, 768), (4, 4096, 8, 768), (1, 320, 5, 15), (3, 2048, 9, 504)])
def test_few_items_balance_compute_units(B, T, H, grid):
    """Persistent forward with fewer than two items per workgroup: workgroups w, w + 256, w + 512
    start on one compute unit, and the causal work of any of them is at most the mean of the busy
    units plus a quarter of the longest block and a tile; run on the host, the decode is shared with the device code."""
    items = M.forward_items(B, T, H, 64, grid)
    nblk = -(-T // 128)
    assert set(map(tuple, items[:, 1:].tolist())) == {(p, b) for p in range(B * H) for b in range(nblk)}
    work = np.bincount(items[:, 0] % 256, weights=items[:, 2] + 1)
    assert work.max() <= work.sum() / len(work) + nblk / 4 + 1
