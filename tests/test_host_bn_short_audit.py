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
]


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
    assert ranges is not None


def test_long_segments_are_not_for_these():
    assert _play((16, 17, 2, 4), (1, 16, 272, 544), 0, 1024, 16)[0] == -2
