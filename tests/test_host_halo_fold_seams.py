"""Reverse exchanges whose lines of ranks are no grid: an open line beside a ring has fewer seams (on the CPU, through the launch
audit)."""
import ctypes

import numpy as np
import pytest
import torch

from dihydrogen_amd import capi
from helpers import CopyAudit


@pytest.mark.parametrize("rows", [100, 4096])
@pytest.mark.parametrize("ring_first", [False, True])
def test_an_open_line_beside_a_ring(ring_first, rows):
    local, w = 6, 2
    peers = [(-1, 1), (0, -1), (3, 3), (2, 2)]  # an open line and a ring
    if ring_first:
        peers = [(1, 1), (0, 0), (-1, 3), (2, -1)]
    with CopyAudit() as audit:
        ts = [torch.zeros(rows, local + 2 * w) for _ in peers]
        for t in ts:
            audit.register(t)
        ranks = (capi.HaloGridRank * len(ts))()
        for k, t, (lower, upper) in zip(ranks, ts, peers):
            k.tensor = t.data_ptr()
            k.local_shape[:4] = local, rows, 1, 1
            for d in range(4):
                k.peer[d][:] = [lower, upper] if d == 0 else [-1, -1]
        grid = capi.HaloGrid(4, len(ts))
        grid.overlap[0], grid.ranks = w, ranks
        assert capi.load().h2x_halo_grid_fold(capi.F32, ctypes.byref(grid), capi.HALO_SUM, None) == 0
    assert (audit.report.outside_loads, audit.report.outside_stores, audit.report.misaligned) == (0, 0, 0)
    for t, (lower, upper) in zip(ts, peers):
        stored, read = np.zeros(t.shape), np.zeros(t.shape)
        stored[:, w:2 * w] += lower >= 0
        stored[:, local:local + w] += upper >= 0
        read[:, :w] += lower >= 0
        read[:, local + w:] += upper >= 0
        loads, stores = audit.counts(t)
        assert np.array_equal(stores, stored.ravel()) and np.array_equal(loads, (stored + read).ravel())
