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
