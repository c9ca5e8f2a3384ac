"""The elements that the workgroups which hold short segments of doubles touch (h2x_bn_audit_short plays the kernels' own
indexing): every interior element counts once, in the range of samples that the staged reduction adds it in, and nothing
outside the interior is stored."""
import ctypes

import numpy as np
import pytest

from dihydrogen_amd import capi
from test_host_bn_ordered_audit import _geometry

# local shape (innermost first), strides: C, N last
CASES = [
    ((7, 7, 5, 9), (1, 7, 49, 245)),
    ((16, 16, 3, 30), (1, 16, 256, 768)),                  # the longest segment
    ((1, 1, 70, 33), (1, 1, 1, 70)),                       # one element a segment
    ((2, 1, 300, 12), (1, 2, 2, 600)),
    ((1, 9, 4, 17), (1, 3, 33, 132)),                      # haloed rows of one element
    ((4, 4, 4, 3, 40), (1, 6, 36, 216, 648)),              # haloed rows, planes and segments
    ((5, 3, 2, 11, 3), (1, 7, 35, 140, 1540)),
    ((15, 17, 2, 64), (1, 15, 255 * 64, 255)),             # samples inside channels
    ((3, 3, 600, 8), (1, 3, 9, 5400)),
    ((255, 1, 1, 120), (1, 255, 255, 255)),
    ((255, 1, 1, 50), (1, 255, 255, 255)),
]
NOT_HELD = [[((255, 1, 1, 120), (1, 255, 255, 255))]] * 2  # by any workgroup, forward and backward


# threads and vectors of the workgroups that there are, forward and backward
LAUNCHED = [{(256, 4), (512, 4), (256, 8), (512, 8), (1024, 8), (512, 16)},
            {(256, 4), (512, 4), (1024, 4), (256, 8), (512, 8), (1024, 8), (256, 16)}]


def _play(shape, strides, backward, threads, vectors):
    size = sum((e - 1) * s for e, s in zip(shape, strides)) + 1
    counted, stored, rng = np.zeros(size, np.uint8), np.zeros(size, np.uint8), np.zeros(size, np.uint16)
    status = capi.load().h2x_bn_audit_short(shape[-1], ctypes.byref(_geometry(shape, strides)), backward, threads, vectors,
                                            counted.ctypes.data, stored.ctypes.data, rng.ctypes.data, size)
    return status, counted, stored, rng


@pytest.mark.parametrize("backward", [0, 1])
@pytest.mark.parametrize("shape,strides", CASES)
def test_every_element_counts_once_in_the_staged_order(shape, strides, backward):
    at = sum(np.arange(e).reshape([-1] + [1] * i) * s for i, (e, s) in enumerate(zip(shape, strides)))
    ranges = None
    for threads in (256, 512, 1024):
        for vectors in (4, 8, 16):
            status, counted, stored, rng = _play(shape, strides, backward, threads, vectors)
            if (threads, vectors) not in LAUNCHED[backward]:
                assert status == -1
                continue
            if status == -2:  # does not hold a channel
                continue
            assert status == 0
            interior = np.zeros(counted.size, np.uint8)
            interior[at.ravel()] = 1
            assert np.array_equal(counted, interior) and np.array_equal(stored, interior)
            if ranges is None:
                ranges = rng
                of_sample = np.asarray([rng[n * strides[-1]] for n in range(shape[-1])], np.int64)
                # ranges of as many neighbouring samples, the last one of what is left
                per = int((of_sample == 1).sum())
                assert np.array_equal(of_sample, 1 + np.arange(shape[-1]) // per)
                whole = np.broadcast_to(of_sample.reshape([-1] + [1] * (len(shape) - 1)), at.shape)
                assert np.array_equal(rng[at], whole)
            assert np.array_equal(rng, ranges)
    assert (ranges is None) == ((shape, strides) in NOT_HELD[backward])


def test_long_segments_are_not_for_these():
    assert _play((16, 17, 2, 4), (1, 16, 272, 544), 0, 1024, 16)[0] == -2


@pytest.mark.parametrize("dims", [2, 3])
def test_every_halo_cell_is_cleared_and_no_other(dims):
    """Boxes with uneven and one-sided halos."""
    rnd = np.random.RandomState(dims)
    lib = capi.load()
    for _ in range(400):
        local, lower, upper = (rnd.randint(lo, hi, dims) for lo, hi in ((1, 8), (0, 4), (0, 4)))
        n, c = rnd.randint(1, 4, 2)
        g = capi.HaloedGeometry()
        g.num_dims = dims + 2
        for d in range(dims):
            g.local_shape[d], g.real_shape[d], g.lower_halo[d] = local[d], local[d] + lower[d] + upper[d], lower[d]
        for d, e in ((dims, c), (dims + 1, n)):
            g.local_shape[d] = g.real_shape[d] = e
        want = np.ones([n, c] + [l + lo + up for l, lo, up in zip(local, lower, upper)][::-1], np.uint8)
        want[(Ellipsis,) + tuple(slice(lo, lo + l) for l, lo in zip(local, lower))[::-1]] = 0
        cleared = np.zeros(want.size, np.uint8)
        threads = int(rnd.choice([1, 7, 256, 1024]))
        assert lib.h2x_bn_audit_cleared(ctypes.byref(g), threads, cleared.ctypes.data, cleared.size) == 0
        assert np.array_equal(cleared, want.ravel()), (local, lower, upper, n, c)
