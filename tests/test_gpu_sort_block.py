"""The routing sort at one block of 1024 assignments, which counts for itself, and one
past it, against the oracle; indices of other ranks' experts included."""

import numpy as np
import pytest
import torch

import nanopysche_amd as fm
from oracle import routing as orouting

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A", [1, 63, 257, 1023, 1024, 1025])
@pytest.mark.parametrize("E,lo,hi", [(1, 0, 1), (8, 0, 8), (256, 0, 256), (32, -5, 40)])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_one_block(dev, A, E, lo, hi, dtype):
    idx = torch.randint(lo, hi, (A, 1), generator=torch.Generator().manual_seed(A + E))
    plan = fm.route_tokens(idx.to(dtype).to(dev), E, 3)
    inside = (idx >= 0) & (idx < E)
    kept = idx[inside].numpy()
    counts = np.bincount(kept, minlength=E)
    assert plan.counts.tolist() == counts.tolist()
    assert plan.use_fp8.tolist() == (counts >= 3).astype(int).tolist()
    offsets = np.concatenate(([0], np.cumsum((counts + 127) // 128 * 128)))
    assert plan.offsets.tolist() == offsets.tolist()
    rows = torch.full((A,), -1, dtype=torch.int64)
    nxt = offsets.copy()
    slots = np.full(plan.rows_max, -1)
    for a in range(A):   # stable: assignment order within an expert
        if bool(inside[a]):
            e = int(idx[a])
            rows[a] = nxt[e]
            slots[nxt[e]] = a
            nxt[e] += 1
    assert plan.row_of.flatten().tolist() == rows.tolist()
    assert plan.assign_of_row.tolist() == slots.tolist()
    if lo == 0:
        ref = orouting.sort_assignments(idx.numpy(), E)
        assert np.array_equal(plan.offsets.cpu().numpy(), ref["offsets"])
