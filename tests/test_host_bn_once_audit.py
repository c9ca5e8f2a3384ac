"""The elements that workgroups holding channels in registers touch (h2x_bn_audit_once plays the
kernels' own indexing): every interior element counts once, nothing outside the interior is stored."""
import ctypes

import numpy as np
import pytest

from dihydrogen_amd import capi

# local shape (innermost first), strides
CASES = [
    ((49, 3, 5), (1, 49, 147)),                                   # segments of no whole number of vectors
    ((4, 2, 3), (1, 4, 8)),                                       # one float vector a segment
    ((7, 7, 6, 4), (1, 7, 49, 294)),
    ((30, 3, 5, 4, 2), (1, 32, 160, 1120, 4480)),                 # haloed rows, planes and segments
    ((5, 9, 2, 3), (1, 7, 80, 170)),                              # rows longer than a vector by one, loose strides
    ((6, 1, 4, 2, 3), (1, 6, 8, 40, 100)),                        # planes of one row with gaps between them
    ((33, 35, 2, 2, 2), (1, 37, 1443, 5772, 11544)),
    ((8, 4, 3, 5), (1, 8, 160, 32)),                              # samples inside channels
]


@pytest.mark.parametrize("member_vectors", [0, 4, 256])
@pytest.mark.parametrize("shape,strides", CASES)
def test_every_element_counts_once(shape, strides, member_vectors):
    g = capi.TensorGeometry()
    g.num_dims = len(shape)
    for i, (e, s) in enumerate(zip(shape, strides)):
        g.local_shape[i], g.strides[i] = e, s
    size = sum((e - 1) * s for e, s in zip(shape, strides)) + 1
    counted, stored = np.zeros(size, np.uint8), np.zeros(size, np.uint8)
    status = capi.load().h2x_bn_audit_once(shape[-1], ctypes.byref(g), member_vectors,
                                           counted.ctypes.data, stored.ctypes.data, size)
    assert status == 0
    at = sum(np.arange(e).reshape([-1] + [1] * i) * s for i, (e, s) in enumerate(zip(shape, strides)))
    interior = np.zeros(size, np.uint8)
    interior[at.ravel()] = 1
    assert np.array_equal(counted, interior) and np.array_equal(stored, interior)


def test_rows_below_a_vector_are_not_taken():
    g = capi.TensorGeometry()
    g.num_dims = 4
    for i, (e, s) in enumerate(zip((3, 5, 2, 2), (1, 4, 20, 40))):
        g.local_shape[i], g.strides[i] = e, s
    b = np.zeros(80, np.uint8)
    assert capi.load().h2x_bn_audit_once(2, ctypes.byref(g), 0, b.ctypes.data, b.ctypes.data, 80) == -2  # unsupported
