"""Receive buffers asked for only after an exchange that went straight from tensor to tensor, against those that
the packed exchange fills as it goes."""
import pytest

import test_host_direct_launch_audit as audits
from test_gpu_direct import _tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("is_reverse", [False, True])
@pytest.mark.parametrize("case", audits.GRIDS)
def test_buffers_after_an_exchange(case, is_reverse):
    """Equal, but for the cells that a later dimension's phase has written since: its halos, or in the
    reverse exchange the boundary cells that its halos were added to."""
    import torch
    from dihydrogen_amd import capi
    from dihydrogen_amd.layers import HaloExchangeAccumOp, HaloExchangeVirtual
    shape, locale, overlap = case
    a, b = (_tensors(shape, locale, None, overlap, torch.float32, 11) for _ in range(2))
    xa, xb = HaloExchangeVirtual(a, periodic=True), HaloExchangeVirtual(b, periodic=True)
    if not xa._grid(2 if is_reverse else 1):
        pytest.skip("boundary strips that share cells: packed on both sides")
    xb._grid_of = (xb._addresses(), 0, -1)      # as where the tensors do not share a GPU
    for x in (xa, xb):
        x.exchange(is_reverse=is_reverse, op=HaloExchangeAccumOp.SUM if is_reverse else HaloExchangeAccumOp.ID)
    assert not xa._recv and xb._recv
    for (r, dim, side), want in xb._recv.items():
        got = xa.recv_buffer(r, dim, side)
        extents = list(a[r].local_real_shape)
        extents[dim] = overlap[dim]
        same = torch.ones(extents[::-1], dtype=torch.bool, device="cuda")
        for d in range(dim + 1, len(extents)):
            w, n = xa.dist.overlap[d], extents[d]
            if w:
                first = w if is_reverse else 0
                axis = len(extents) - 1 - d
                same.narrow(axis, first, w).fill_(False)
                same.narrow(axis, n - first - w, w).fill_(False)
        same = same.ravel()
        assert torch.equal(got[same], want[same]), (r, dim, side)


def test_buffers_packed_on_a_stream_of_the_exchange_are_there_for_the_current_one():
    """Asked for after the exchange's own stream has been waited for: what is packed then is waited for as well."""
    import torch
    from dihydrogen_amd import capi
    from dihydrogen_amd.layers import HaloExchangeVirtual
    side = torch.cuda.Stream()
    ts = _tensors((512, 300, 32, 2), (2, 1, 1, 1), None, (1, 0, 0, 0), torch.float32, 3)
    want = ts[0].interior_view()[..., -1].flatten().clone()
    torch.cuda.synchronize()
    xch = HaloExchangeVirtual(ts, stream=side)
    xch.exchange()
    side.synchronize()
    busy = torch.empty(1 << 26, device="cuda")
    with torch.cuda.stream(side):
        for _ in range(20):     # the packing waits behind some milliseconds
            busy.normal_()
    assert torch.equal(xch.recv_buffer(1, 0, capi.LHS), want)
