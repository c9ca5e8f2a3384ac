"""Which halo exchanges go straight from tensor to tensor, and that the others are done (or refused) as
strips through buffers - on the CPU, through the launch audit of the copy entry points."""
import numpy as np
import pytest

import test_host_copy_launch_audit as packed
from helpers import CopyAudit


@pytest.fixture(autouse=True)
def direct(monkeypatch):
    from dihydrogen_amd import layers
    monkeypatch.setattr(layers, "_share_a_gpu", lambda tensors: True)


@pytest.mark.parametrize("widths", [(2, 1), (1, 2)])
def test_ranks_with_halos_of_unequal_widths(widths):
    """An exchange at the first rank's width: refused where another rank's halo is narrower, and within the
    strips of every rank where it is wider."""
    from dihydrogen_amd.layers import HaloExchangeVirtual
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    with CopyAudit() as audit:
        ts = []
        for r, w in enumerate(widths):
            dist = Distribution.make_overlapped_distribution([2, 1, 1, 1], [w, 0, 0, 0])
            ts.append(Tensor([12, 5, 2, 1], LocaleVirtual(r, 2), dist, device="cpu").allocate())
            audit.register(ts[-1].data)
        xch = HaloExchangeVirtual(ts)
        if widths[1] < widths[0]:
            with pytest.raises(ValueError, match="exceeds the overlap"):
                xch.exchange()
            with pytest.raises(ValueError, match="exceeds the overlap"):
                xch.exchange(is_reverse=True)
        else:
            xch.exchange()
            assert audit.buffers
        xch.clear_halos()
    packed._clean(audit.report)
    for t in ts:
        assert np.array_equal(audit.counts(t.data)[1] > 0, packed._strip(t, 0, 0, t.overlap[0], inner=False).ravel()
                              | packed._strip(t, 0, 1, t.overlap[0], inner=False).ravel())


@pytest.mark.parametrize("status", [-2, -3])
@pytest.mark.parametrize("step", ["forward", "reverse", "clear"])
def test_what_the_whole_grid_launches_refuse_goes_through_buffers(step, status, monkeypatch):
    import torch
    from dihydrogen_amd import layers
    shape, locale, overlap = packed.HALO_CASES[1]
    results = []
    for refuse in (False, True):
        with CopyAudit() as audit:
            ts = packed._tensors(shape, locale, overlap, torch.float32, audit)
            xch = layers.HaloExchangeVirtual(ts)
            if refuse:
                calls = xch._calls

                class Refusing:
                    def __getattr__(self, name):
                        return (lambda *args: status) if name.startswith("h2x_halo_grid_") else getattr(calls, name)

                xch._calls = Refusing()
            if step == "clear":
                xch.clear_halos()
            else:
                xch.exchange(is_reverse=step == "reverse")
        packed._clean(audit.report)
        assert bool(audit.buffers) == (refuse and step != "clear")
        results.append([audit.counts(t.data)[1] > 0 for t in ts])
    for a, b in zip(*results):
        assert np.array_equal(a, b)


def test_limits_of_a_reverse_exchange_are_those_of_one_rank_and_of_a_launch():
    """Ranks of short rows, imaginary addresses: what is not refused fails for want of a GPU.  A launch
    has up to 2^32 - 1 threads, one a row here, and one rank up to 2^31."""
    import ctypes

    import torch
    from dihydrogen_amd import capi
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible: these calls would launch on imaginary pointers")

    def fold(num_ranks, rows):
        ranks = (capi.HaloGridRank * num_ranks)()
        for r, k in enumerate(ranks):
            k.tensor = 1 << 20
            k.local_shape[:4] = 2, rows, 1, 1
            for d in range(4):
                k.peer[d][:] = [(r - 1) % num_ranks, (r + 1) % num_ranks] if d == 0 else [-1, -1]
        grid = capi.HaloGrid(4, num_ranks)
        grid.overlap[0], grid.ranks = 1, ranks
        return capi.load().h2x_halo_grid_fold(capi.F32, ctypes.byref(grid), capi.HALO_SUM, None)

    assert fold(8, 1000) > 0
    assert fold(8, 270_000_000) > 0                # 2.16 billion threads
    assert fold(16, 256 * (0xffffff // 16)) > 0    # 4.29 billion
    assert fold(16, 256 * (0xffffff // 16) + 1) == capi.ERR_TOO_LARGE
    assert fold(2, 536_870_912) == capi.ERR_TOO_LARGE  # tensors of 2^31 elements


@pytest.mark.parametrize("step", ["forward", "reverse", "clear"])
def test_samples_spread_unevenly_over_the_ranks(step):
    """Space and samples are both distributed: neighbours hold the same samples, other ranks fewer."""
    import torch
    from dihydrogen_amd import capi
    from dihydrogen_amd.layers import HaloExchangeVirtual
    with CopyAudit() as audit:
        ts = packed._tensors((12, 10, 2, 3), (2, 2, 1, 2), (1, 1, 0, 0), torch.float32, audit)
        assert len({t.local_shape[3] for t in ts}) == 2
        xch = HaloExchangeVirtual(ts)
        if step == "clear":
            xch.clear_halos()
        else:
            xch.exchange(is_reverse=step == "reverse")
    packed._clean(audit.report)
    for r, t in enumerate(ts):
        if step == "clear":
            want = np.any([packed._strip(t, d, side, 1, inner=False) for d in (0, 1) for side in (capi.LHS, capi.RHS)],
                          axis=0).ravel()
        else:
            want = packed._expected_exchange(xch, reverse=step == "reverse")[1][r] > 0
        assert np.array_equal(audit.counts(t.data)[1] > 0, want)


@pytest.mark.parametrize("is_reverse", [False, True])
def test_a_receive_buffer_asked_for_after_an_exchange_holds_its_strip(is_reverse):
    """Exchanged straight from tensor to tensor, packed when a buffer is asked for, and by the next exchange itself."""
    import torch
    from dihydrogen_amd import capi
    from dihydrogen_amd.layers import HaloExchangeVirtual
    shape, locale, overlap = packed.HALO_CASES[4]
    with CopyAudit() as audit:
        ts = packed._tensors(shape, locale, overlap, torch.float32, audit)
        xch = HaloExchangeVirtual(ts)
        xch.exchange(is_reverse=is_reverse)
        assert not audit.buffers
        expected = [(r, d, s) for r in range(8) for d in range(3) for s in (capi.LHS, capi.RHS)
                    if xch.find_peer_rank(r, d, s) is not None]
        first = {key: xch.recv_buffer(*key) for key in expected}
        written = {key: audit.counts(b) for key, b in first.items()}
        for loads, stores in written.values():
            assert (stores == 1).all() and not loads.any()
        xch.exchange(is_reverse=is_reverse)
        for key in expected:
            assert xch.recv_buffer(*key).data_ptr() == first[key].data_ptr()
            loads, stores = audit.counts(first[key])
            assert (stores == 2).all() and (loads == 1).all()
    packed._clean(audit.report)


def test_strips_packed_since_an_exchange_are_not_packed_again():
    import torch
    from dihydrogen_amd import capi
    from dihydrogen_amd.layers import HaloExchangeVirtual
    shape, locale, overlap = packed.HALO_CASES[0]
    with CopyAudit() as audit:
        ts = packed._tensors(shape, locale, overlap, torch.float32, audit)
        xch = HaloExchangeVirtual(ts)
        xch.exchange()
        for _ in range(3):
            xch.exchange_dim(0, 1, 1, 1, 1)
        assert xch._packed_since == (0,)        # noted once, however often it is packed
        xch.exchange(fused=True)
        for dim in (0, 1):
            loads, stores = audit.counts(xch.recv_buffer(0, dim, capi.RHS))
            assert (stores == (3, 1)[dim]).all() and (loads == (3, 0)[dim]).all()
        ts[0].data = ts[0].data.clone()
        other = HaloExchangeVirtual(ts)
        other._direct = ((0,) * 4, False)      # exchanged when the tensors lay elsewhere
        with pytest.raises(RuntimeError, match="reallocated"):
            other.recv_buffer(0, 0, capi.RHS)
