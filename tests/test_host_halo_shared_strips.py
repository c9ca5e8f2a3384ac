"""Reverse exchanges of ranks whose two boundary strips share cells: the strips are combined one after the other.
On the CPU, through the launch audit of the copy entry points."""
import numpy as np
import pytest

import test_host_copy_launch_audit as packed
from helpers import CopyAudit

# ranks of 1 and 2 cells with halos of 1; of 3 cells with halos of 2; of 2 and 3 cells, where the exchange is one launch
CASES = [((5, 4, 2, 1), (3, 1, 1, 1), (1, 0, 0, 0), 2), ((4, 9, 2, 1), (1, 3, 1, 1), (0, 2, 0, 0), 2),
         ((8, 4, 2, 1), (3, 1, 1, 1), (1, 0, 0, 0), 1)]


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("shape,locale,overlap,launches", CASES)
def test_strips_that_share_cells_take_two_launches(shape, locale, overlap, launches, fused):
    import torch
    from dihydrogen_amd.layers import HaloExchangeAccumOp, HaloExchangeVirtual
    for dtype in (torch.float32, torch.float64):
        with CopyAudit() as audit:
            ts = packed._tensors(shape, locale, overlap, dtype, audit)
            xch = HaloExchangeVirtual(ts, periodic=True)
            xch.exchange(is_reverse=True, op=HaloExchangeAccumOp.SUM, fused=fused)
            halo, boundary = packed._expected_exchange(xch, reverse=True)
        packed._clean(audit.report)
        assert audit.report.launches == launches + (not fused)
        for t, h, b in zip(ts, halo, boundary):
            loads, stores = audit.counts(t.data)
            assert np.array_equal(loads, h + b) and np.array_equal(stores, b)


@pytest.mark.parametrize("is_reverse", [False, True])
@pytest.mark.parametrize("shape,locale,overlap", [((5, 9, 2, 1), (3, 2, 1, 1), (2, 2, 0, 0)), ((5, 9, 2, 1), (1, 5, 1, 1), (0, 3, 0, 0))])
def test_ranks_narrower_than_a_halo_are_exchanged_through_buffers(shape, locale, overlap, is_reverse):
    """Their boundary strips reach into the halos that the same phase writes: everything is read first."""
    import torch
    from dihydrogen_amd.layers import HaloExchangeVirtual
    results = []
    for fused in (True, False):
        with CopyAudit() as audit:
            ts = packed._tensors(shape, locale, overlap, torch.float32, audit)
            HaloExchangeVirtual(ts, periodic=True).exchange(is_reverse=is_reverse, fused=fused)
        packed._clean(audit.report)
        assert audit.buffers
        for b in audit.buffers:
            loads, stores = audit.counts(b)
            assert (loads == 1).all() and (stores == 1).all()
        results.append([np.stack(audit.counts(t.data)) for t in ts])
    for a, b in zip(*results):
        assert np.array_equal(a, b)
