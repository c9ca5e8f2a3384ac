"""The elements that the workgroups which read double tensors once touch (h2x_bn_audit_ordered plays the
kernels' own indexing): every interior element counts once, in the sum of the staged workgroup that
adds it in the two-launch calls, and nothing outside the interior is stored."""
import ctypes

import numpy as np
import pytest

from dihydrogen_amd import capi

# local shape (innermost first), strides: C, N last
CASES = [
    ((56, 56, 3, 5), (1, 56, 3136, 9408)),                        # aligned whole vectors
    ((33, 33, 33, 2, 3), (1, 33, 1089, 35937, 71874)),            # segments of an odd length: one row each
    ((17, 17, 2, 9), (1, 17, 289, 578)),                          # segments of 257 to 1023: samples are folded
    ((300, 3, 7), (1, 300, 900)),
    ((30, 30, 30, 2, 2), (1, 32, 1024, 32768, 65536)),            # haloed rows, planes and segments
    ((33, 35, 2, 2, 2), (1, 37, 1443, 5772, 11544)),
    ((128, 20, 3, 2), (1, 128, 16000, 3000)),                     # samples inside channels
    ((2, 700, 2, 3), (1, 5, 3600, 7300)),                         # rows of one vector
    ((2049, 2, 3), (1, 2049, 4098)),                              # one element beyond a tile
    ((256, 16, 1, 70), (1, 256, 4096, 4096)),                     # more units than groups of a budget
]


def _geometry(shape, strides):
    g = capi.TensorGeometry()
    g.num_dims = len(shape)
    for i, (e, s) in enumerate(zip(shape, strides)):
        g.local_shape[i], g.strides[i] = e, s
    return g


def _play(shape, strides, backward, passes):
    size = sum((e - 1) * s for e, s in zip(shape, strides)) + 1
    counted, stored, group = np.zeros(size, np.uint8), np.zeros(size, np.uint8), np.zeros(size, np.uint16)
    g = _geometry(shape, strides)
    status = capi.load().h2x_bn_audit_ordered(shape[-1], ctypes.byref(g), backward, passes, counted.ctypes.data,
                                              stored.ctypes.data, group.ctypes.data, size)
    return status, counted, stored, group


@pytest.mark.parametrize("passes", [1, 2, 4])
@pytest.mark.parametrize("backward", [0, 1])
@pytest.mark.parametrize("shape,strides", CASES)
def test_every_element_counts_once_in_the_staged_order(shape, strides, backward, passes):
    status, counted, stored, group = _play(shape, strides, backward, passes)
    assert status == 0
    at = sum(np.arange(e).reshape([-1] + [1] * i) * s for i, (e, s) in enumerate(zip(shape, strides)))
    interior = np.zeros(counted.size, np.uint8)
    interior[at.ravel()] = 1
    assert np.array_equal(counted, interior) and np.array_equal(stored, interior)
    assert np.array_equal(group > 0, interior > 0)
    # however many groups a member plays, an element belongs to the same one
    assert np.array_equal(group, _play(shape, strides, backward, 1)[3])


@pytest.mark.parametrize("shape,strides", [((16, 16, 5, 4), (1, 16, 256, 1280)),     # short segments
                                           ((1, 900, 2, 2), (1, 3, 2700, 5400)),     # rows below a vector
                                           ((64, 64, 64, 4, 64), (1, 64, 4096, 262144, 1048576))])  # too many groups or offsets
def test_what_runs_in_two_launches(shape, strides):
    for backward in (0, 1):
        b = (ctypes.c_ubyte * 16)()
        status = capi.load().h2x_bn_audit_ordered(shape[-1], ctypes.byref(_geometry(shape, strides)), backward, 1, b, b, b, 16)
        assert status == -2  # unsupported: played into 16 bytes, what is supported gives -1


@pytest.mark.parametrize("case,needed", [((8, 32, 33, 33, 33), True), ((8, 64, 1, 56, 56), True), ((1, 200, 1, 40, 40), False),
                                         ((64, 512, 1, 14, 14), False), ((100, 64, 64, 64, 64), False)])
def test_state_of_double_tensors(case, needed):
    n, c, d, h, w = case
    shape, strides, at = (w, h, d, c, n), [], 1
    for e in shape:
        strides.append(at)
        at *= e
    lib = capi.load()
    got = lib.h2x_bn_ordered_state_needed(n, ctypes.byref(_geometry(shape, strides)))
    assert got == (lib.h2x_bn_team_state_bytes(c) if needed else 0)


@pytest.mark.parametrize("backward", [0, 1])
@pytest.mark.parametrize("n,units", [(9, 1), (8, 1), (17, 1), (5, 3), (12, 2)])
def test_no_more_groups_than_the_units_of_the_busiest_need(n, units, backward):
    """A place of a team that a group leaves empty is an idle one: of 600 channels, which are cut into 8 groups at most."""
    c, h, w = 600, 40, 30 + 52 * (units - 1)
    status, counted, _, group = _play((w, h, c, n), (1, w, w * h, w * h * c), backward, 1)
    assert status == 0
    first = group.reshape(n, c, h * w)[:, 0]                     # of the first channel
    played = np.zeros(int(first.max()) + 1, np.int64)
    for sample in first:
        for u in range(units):
            played[sample[u * 2048]] += 1
    assert played.sum() == n * units and played[0] == 0
    busiest, groups = played.max(), len(played) - 1
    assert groups <= 8 and groups * busiest - n * units < busiest


@pytest.mark.parametrize("n,c,h,w,halo", [(160, 133, 23, 19, 1), (184, 91, 23, 26, 1), (231, 51, 48, 12, 1)])
def test_two_launches_where_members_are_mostly_padding(n, c, h, w, halo):
    """Units of 2048 elements of which a segment's rows fill a third: teams of them take 1.1 to 1.5 times as long."""
    lib, pitch = capi.load(), w + 2 * halo
    plane = pitch * (h + 2 * halo)
    assert lib.h2x_bn_ordered_state_needed(n, ctypes.byref(_geometry((w, h, c, n), (1, pitch, plane, plane * c)))) == 0
