"""What the launches that go straight from tensor to tensor touch (halo exchange, reverse exchange and
clearing of a whole grid of ranks, shuffle without an arena) - on the CPU, through the launch audit of the
copy entry points.  Expectations come from the definition of strips and boxes.  A vector at the end of a
run may move a few elements twice, so cells are counted as touched or not, except where elements are
accumulated: those are read and written exactly as often as a strip covers them."""
import itertools

import numpy as np
import pytest

import test_host_copy_launch_audit as packed
from helpers import CopyAudit

GRIDS = packed.HALO_CASES + [
    ((9, 7, 2, 1), (3, 2, 1, 1), (1, 1, 0, 0)),             # rows of three cells: shorter than a vector
    ((10, 10, 10, 3, 2), (2, 2, 2, 1, 1), (2, 1, 2, 0, 0)),
    ((6, 8, 13, 3, 1), (1, 2, 3, 1, 1), (0, 2, 1, 0, 0)),   # no halo along the rows, ranks of unequal extents
    ((600, 20, 1, 1), (2, 2, 1, 1), (5, 2, 0, 0)),          # ends of more than a vector, more than a workgroup of rows
    ((8, 12, 2, 1), (4, 4, 1, 1), (1, 1, 0, 0)),            # 16 ranks, interiors of exactly two halos
]


@pytest.fixture(autouse=True)
def direct(monkeypatch):
    from dihydrogen_amd import layers
    monkeypatch.setattr(layers, "_share_a_gpu", lambda tensors: True)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("step", ["forward", "reverse", "clear", "clear unfilled"])
def test_a_grid_of_ranks_touches_the_strips_and_nothing_else(step, periodic, dtype):
    import torch
    from dihydrogen_amd import capi
    from dihydrogen_amd.layers import HaloExchangeAccumOp, HaloExchangeVirtual
    for shape, locale, overlap in GRIDS:
        with CopyAudit() as audit:
            ts = packed._tensors(shape, locale, overlap, getattr(torch, dtype), audit)
            xch = HaloExchangeVirtual(ts, periodic=periodic)
            assert xch._grid(1)
            if step == "reverse" and not xch._grid(2):
                continue    # boundary strips that share cells are folded one after the other
            if step == "forward":
                xch.exchange()
            elif step == "reverse":
                xch.exchange(is_reverse=True, op=HaloExchangeAccumOp.SUM)
            else:
                xch.clear_halos(only_unfilled=step == "clear unfilled")
        assert not audit.buffers
        assert (audit.report.outside_loads, audit.report.outside_stores, audit.report.misaligned) == (0, 0, 0)
        assert audit.report.launches <= (sum(o > 0 for o in overlap) if step == "reverse" else 1)
        inner, outer = packed._expected_exchange(xch, reverse=False)
        for r, t in enumerate(ts):
            what = (shape, locale, overlap, step, periodic, r)
            loads, stores = audit.counts(t.data)
            if step == "forward":
                assert np.array_equal(stores > 0, outer[r] > 0), what
                assert not loads[outer[r] > 0].any(), what    # no cell is read that this launch writes
            elif step == "reverse":
                assert np.array_equal(loads, inner[r] + outer[r]) and np.array_equal(stores, inner[r]), what
            else:
                want = np.zeros(t.local_real_shape[::-1], bool)
                for d, side in itertools.product(range(xch.nd), (capi.LHS, capi.RHS)):
                    if t.overlap[d] and not (step == "clear unfilled" and xch.find_peer_rank(r, d, side) is not None):
                        want |= packed._strip(t, d, side, t.overlap[d], inner=False)
                assert np.array_equal(stores > 0, want.ravel()) and not loads.any(), what


@pytest.mark.parametrize("dtype", ["float32", "int16", "float64"])
def test_a_direct_shuffle_moves_every_element(dtype):
    import torch
    import test_gpu_shuffle as cases
    from dihydrogen_amd.layers import TensorShufflerVirtual
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    extra = {"elements": ((3, 5, 4, 1, 1), ([3, 1, 1, 1, 1], None, [1, 0, 0, 0, 0]), ([1, 1, 3, 1, 1], None, None)),
             "unequal": ((37, 3, 9, 5), ([1, 1, 1, 4], None, None), ([2, 1, 2, 1], None, [1, 0, 0, 0]))}
    for (name, (shape, (sl, ss, so), (dl, ds, do))), forward in itertools.product({**cases.CASES, **extra}.items(),
                                                                                  (True, False)):
        n = int(np.prod(sl))
        with CopyAudit() as audit:
            make = lambda l, s, o: [Tensor(shape, LocaleVirtual(r, n), Distribution(l, s, o), getattr(torch, dtype),
                                           device="cpu").allocate() for r in range(n)]
            src, dst = make(sl, ss, so), make(dl, ds, do)
            for t in src + dst:
                audit.register(t.data)
            sh = TensorShufflerVirtual(src, dst)
            assert sh._direct_plan is not None, name
            (sh.shuffle_forward if forward else sh.shuffle_backward)()
            del sh
        packed._clean(audit.report)
        assert not audit.buffers and audit.report.launches == 1, name
        read = src if forward else dst
        for t in src + dst:
            want = np.zeros(t.local_real_shape[::-1], bool)
            if t.is_split_root():
                want[tuple(slice(o, o + l) for o, l in zip(reversed(t.overlap), reversed(t.local_shape)))] = True
            loads, stores = audit.counts(t.data)
            moved, other = (loads, stores) if any(t is q for q in read) else (stores, loads)
            assert not other.any(), (name, forward)
            assert np.array_equal(moved > 0, want.ravel()) if want.size else not moved.any(), (name, forward)
