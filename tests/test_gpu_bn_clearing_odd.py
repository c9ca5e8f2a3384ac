"""Whole batch-norm passes that clear the halo, where a segment of the allocation is no whole number of vectors:
its last vector starts early, within the halo."""
import ctypes

import pytest

import test_gpu_bn_once as once
from dihydrogen_amd import capi

pytestmark = pytest.mark.gpu


# 2 to 601 channels by one workgroup and by teams; 1, 2 and 3 elements beyond whole vectors
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("shape,halo", [((1, 2, 1, 5, 5), 1), ((3, 5, 9, 9, 9), 1), ((2, 4, 1, 55, 27), 3),
                                        ((2, 4, 1, 1, 3), 1), ((7, 601, 1, 37, 32), 1), ((2, 40, 31, 31, 31), 1),
                                        ((9, 33, 21, 19, 18), 2), ((5, 3, 1, 175, 201), 2)])
def test_as_the_staged_calls(shape, halo, in_place):
    once.test_whole_pass_that_clears_the_halo(shape, halo, in_place)


@pytest.mark.parametrize("width,status", [(9, -2), (10, 0), (7, -2)])
def test_a_last_vector_with_interior_cells_is_refused(width, status):
    """Halos of 1 along the rows only: one cell behind the interior."""
    import torch
    n, c, h = 3, 4, 5
    g = capi.HaloedGeometry()
    g.num_dims = 4
    for i, (e, o) in enumerate(zip((width, h, c, n), (1, 0, 0, 0))):
        g.local_shape[i], g.real_shape[i], g.lower_halo[i] = e, e + 2 * o, o
    x, y = (torch.zeros(n, c, h, width + 2, device="cuda") for _ in range(2))
    state = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    v = [torch.ones(c, device="cuda") for _ in range(6)]
    a = lambda t: t.data_ptr()
    assert capi.load().h2x_bn_forward_clearing(capi.F32, ctypes.byref(g), a(x), a(v[0]), a(v[1]), n * h * width, 0.9, 1e-5,
                                               *[a(t) for t in v[2:]], a(y), a(state), None) == status
    torch.cuda.synchronize()
