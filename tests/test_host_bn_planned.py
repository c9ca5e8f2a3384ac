"""Which kernels the whole batch-norm passes launch (h2x_bn_planned asks the entry points themselves), for the shapes by which the GPU tests
mean to reach them, on the CPU: those compare results only, and would agree as well if a rule sent every call elsewhere."""
import ctypes

import pytest

from dihydrogen_amd import capi
import test_gpu_bn_clearing_doubles as clearing
import test_gpu_bn_shared_statistics as shared
import test_gpu_bn_short_ordered as short
import test_gpu_bn_windows as windows

ONCE, WINDOW, TEAM, ORDERED, ORDERED_TEAM, SHORT = 8, 9, 10, 11, 12, 13
TWO_LAUNCHES = [0, 1], [2, 3]  # forward, backward


def _geometry(local, real):
    """Both innermost first, samples last."""
    g = capi.TensorGeometry()
    g.num_dims, stride = len(local), 1
    for d, (e, r) in enumerate(zip(local, real)):
        g.local_shape[d], g.strides[d] = e, stride
        stride *= r
    return g


def _haloed(local, halo):
    h = capi.HaloedGeometry()
    h.num_dims = len(local)
    for d, e in enumerate(local):
        o = halo[d] if d < len(halo) else 0
        h.local_shape[d], h.real_shape[d], h.lower_halo[d] = e, e + 2 * o, o
    return h


def _kernels(backward, dtype, n, geometry=None, cleared=None, state=1):
    """Numbers of the kernels, None for the staged calls."""
    launches, count = (capi.BnPlannedLaunch * capi.BN_AUDIT_MAX_LAUNCHES)(), ctypes.c_int()
    status = capi.load().h2x_bn_planned(backward, dtype, n, geometry and ctypes.byref(geometry), cleared and ctypes.byref(cleared),
                                        state, launches, ctypes.byref(count))
    if status == capi.ERR_UNSUPPORTED:
        return None
    assert status == 0
    return [l.kernel for l in launches[:count.value]]


def _once(dtype, n, c, d, h, w, halo=0):
    hd = halo if d > 1 else 0
    g = _geometry((w, h, d, c, n), (w + 2 * halo, h + 2 * halo, d + 2 * hd, c, n))
    return [_kernels(backward, dtype, n, g) for backward in (0, 1)]


# of the shapes of the windows' test those on the other side of an edge of the rule
NO_WINDOWS = [(156, 701, 1, 7, 7), (157, 700, 1, 7, 7), (313, 512, 1, 7, 7), (64, 1024, 1, 1, 128)]


@pytest.mark.parametrize("shape", windows.SHAPES)
def test_windows(shape):
    assert _once(capi.F32, *shape) == [[ONCE if shape in NO_WINDOWS else WINDOW]] * 2


@pytest.mark.parametrize("n,c,w,pad,kernel", [(128, 1023, 49, 2, WINDOW), (128, 1024, 49, 49, WINDOW), (128, 1024, 49, 50, ONCE)])
def test_windows_of_channels_that_lie_apart(n, c, w, pad, kernel):
    g = _geometry((w, 1, 1, c, n), (w + pad, 1, 1, c, n))
    assert [_kernels(backward, capi.F32, n, g) for backward in (0, 1)] == [[kernel]] * 2


# two samples of a lane too many backward; a workgroup of few lanes backward; reduced as long segments
TWO_BACKWARD = [(30, 3, 1, 16, 16, 0), (120, 276, 1, 9, 14, 0)]
TWO_BOTH_WAYS = [(64, 2, 1, 17, 15, 0)]


@pytest.mark.parametrize("shape", short.SHAPES)
def test_short_segments_of_doubles(shape):
    forward, backward = _once(capi.F64, *shape)
    assert forward == (TWO_LAUNCHES[0] if shape in TWO_BOTH_WAYS else [SHORT])
    assert backward == (TWO_LAUNCHES[1] if shape in TWO_BOTH_WAYS + TWO_BACKWARD else [SHORT])


@pytest.mark.parametrize("n,c,d,h,w,halo,forward", [(112, 10, 5, 4, 6, 0, TWO_LAUNCHES[0]), (83, 27, 1, 10, 11, 1, TWO_LAUNCHES[0]),
                                                    (56, 21, 5, 6, 5, 1, [SHORT]), (139, 70, 1, 9, 7, 0, [SHORT])])
def test_few_workgroups_with_many_samples(n, c, d, h, w, halo, forward):
    assert _once(capi.F64, n, c, d, h, w, halo)[0] == forward


CLEARING = dict(zip([s[:3] for s in clearing.SHAPES], [SHORT] * 5 + [ORDERED_TEAM] * 3 + [ORDERED] * 2 + [ORDERED_TEAM] * 3 + [ORDERED]))


@pytest.mark.parametrize("n,c,spatial,halo", clearing.SHAPES)
def test_doubles_whose_halo_is_cleared(n, c, spatial, halo):
    kernels = [_kernels(backward, capi.F64, n, cleared=_haloed(spatial + (c, n), halo)) for backward in (0, 1)]
    if (n, c, spatial, halo) in clearing.STAGED:
        assert kernels == [None, None]
    else:
        assert kernels == [[CLEARING[n, c, spatial]]] * 2


# N, C, spatial extents, halo; forward and backward: the two sides of each line of clearing_pays
@pytest.mark.parametrize("n,c,spatial,halo,kernels", [
    (176, 910, (2, 3), 1, "11"), (110, 1655, (6, 5), 3, "11"),                         # up to 200 cells of a segment
    (106, 26, (4, 4, 4), 3, "00"), (119, 88, (6, 5, 4), 2, "00"), (43, 107, (4, 5, 5), 3, "11"), (29, 72, (6, 6, 7), 2, "11"),  # few workgroups
    (57, 454, (9, 18), 3, "00"), (83, 183, (13, 9), 3, "11"), (30, 290, (20, 12), 3, "01"),  # the largest ones, in rounds
    (53, 284, (5, 4, 4), 2, "00"), (51, 350, (6, 4, 5), 2, "11"),                      # a little more than a round
    (22, 1078, (12, 20), 3, "00"), (41, 556, (16, 9), 2, "11"), (9, 412, (4, 5, 7), 3, "11"), (17, 482, (14, 16), 2, "11")])  # large outputs
def test_short_segments_whose_halo_is_cleared(n, c, spatial, halo, kernels):
    for backward in (0, 1):
        planned = _kernels(backward, capi.F64, n, cleared=_haloed(spatial + (c, n), (halo,) * len(spatial)))
        assert planned == ([SHORT] if kernels[backward] == "1" else None)


@pytest.mark.parametrize("dtype,n,c,spatial,halo", shared.SHAPES)
def test_shared_statistics_come_by_every_way(dtype, n, c, spatial, halo):
    real = tuple(e + 2 * halo for e in spatial)
    kernels = _kernels(0, capi.F64 if dtype.itemsize == 8 else capi.F32, n, _geometry(spatial + (c, n), real + (c, n)))
    assert kernels == shared.KERNELS[shared.SHAPES.index((dtype, n, c, spatial, halo))]


def test_no_state_no_teams():
    assert _kernels(0, capi.F32, 4, _geometry((64, 64, 64, 64, 4), (64, 64, 64, 64, 4))) == [TEAM]
    assert _kernels(0, capi.F32, 4, _geometry((64, 64, 64, 64, 4), (64, 64, 64, 64, 4)), state=0) == TWO_LAUNCHES[0]
