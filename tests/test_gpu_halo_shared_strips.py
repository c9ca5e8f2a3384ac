"""Reverse exchanges of ranks with less than two halo widths of interior: both neighbours' strips reach the cells that
the boundary strips share.  Whole numbers, so that sums are exact in any order."""
import numpy as np
import pytest

import test_host_halo_shared_strips as host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("shape,locale,overlap,launches", host.CASES + [((517, 300, 40, 1), (1, 200, 1, 1), (0, 1, 0, 0), 2)])
def test_both_strips_are_added(shape, locale, overlap, launches, fused, dtype):
    import torch
    from dihydrogen_amd.layers import HaloExchangeAccumOp, HaloExchangeVirtual
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    dist = Distribution.make_overlapped_distribution(locale, overlap)
    ts = [Tensor(shape, LocaleVirtual(r, dist.num_ranks), dist, getattr(torch, dtype)).allocate()
          for r in range(dist.num_ranks)]
    g = torch.Generator(device="cuda").manual_seed(8)
    for t in ts:
        t.data.random_(-1000, 1000, generator=g)
    dim = int(np.argmax(overlap))
    w, axis, n = overlap[dim], len(shape) - 1 - dim, dist.num_ranks
    strip = lambda a, first: a.narrow(axis, first, w)
    before = [t.real_view().cpu() for t in ts]
    want = [b.clone() for b in before]
    for r, b in enumerate(want):
        extent = b.shape[axis]
        below, above = before[(r - 1) % n], before[(r + 1) % n]
        strip(b, w).add_(strip(below, below.shape[axis] - w))
        strip(b, extent - 2 * w).add_(strip(above, 0))
    HaloExchangeVirtual(ts, periodic=True).exchange(is_reverse=True, op=HaloExchangeAccumOp.SUM, fused=fused)
    torch.cuda.synchronize()
    for t, b in zip(ts, want):
        assert torch.equal(t.real_view().cpu(), b)


@pytest.mark.parametrize("is_reverse", [False, True])
def test_ranks_narrower_than_a_halo(is_reverse):
    import torch
    from dihydrogen_amd.layers import HaloExchangeAccumOp, HaloExchangeVirtual
    from test_gpu_direct import _tensors
    results = []
    for fused in (True, False):
        ts = _tensors((5, 9, 30, 4), (3, 2, 1, 1), None, (2, 2, 0, 0), torch.float32, 2)
        for t in ts:
            t.data.mul_(1000).round_()      # whole numbers: sums are exact
        HaloExchangeVirtual(ts, periodic=True).exchange(
            is_reverse=is_reverse, op=HaloExchangeAccumOp.SUM if is_reverse else HaloExchangeAccumOp.ID, fused=fused)
        results.append([t.data for t in ts])
    for a, b in zip(*results):
        assert torch.equal(a, b)
