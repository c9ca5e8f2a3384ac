"""Batch-norm backward of dense tensors around 48 MiB, from which dy is read past the caches: as the two-launch calls
(doubles bit for bit) on both sides of that size, also where rows are not whole vectors of a channel."""
import pytest

import test_gpu_bn_once as floats
import test_gpu_bn_ordered as doubles

pytestmark = pytest.mark.gpu

# N, C, D, H, W; the first of each exactly 48 MiB, the second a little less
FLOATS = [(4, 48, 1, 256, 256), (4, 47, 1, 256, 256), (134, 60, 1, 38, 38), (138, 60, 1, 38, 38)]
DOUBLES = [(4, 24, 1, 256, 256), (4, 23, 1, 256, 256), (5, 32, 33, 33, 33), (6, 32, 33, 33, 33)]


@pytest.mark.parametrize("shape", FLOATS)
def test_floats(shape):
    p = floats._Problem(*shape)
    floats._close(p.run("once"), p.run("local_strided"))


@pytest.mark.parametrize("shape", DOUBLES)
def test_doubles(shape):
    p = doubles._Problem(*shape)
    doubles._same(p.run("once"), p.run("local_strided"))


# a halo that is cleared: whole allocations of 48 MiB and a little less
@pytest.mark.parametrize("shape,halo", [((4, 48, 1, 254, 254), 1), ((4, 47, 1, 254, 254), 1)])
def test_cleared_halo(shape, halo):
    floats.test_whole_pass_that_clears_the_halo(shape, halo, False)
