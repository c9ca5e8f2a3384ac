"""Batch-norm of a few channels of megabytes, whose teams have members of more than 32 KB however few those are:
as the two-launch calls (doubles bit for bit), around the numbers of workgroups where the rules change."""
import pytest

import test_gpu_bn_once as floats
import test_gpu_bn_ordered as doubles

pytestmark = pytest.mark.gpu

# N, C, D, H, W
FLOATS = [(1, 2, 90, 90, 90), (2, 1, 96, 96, 96), (3, 3, 64, 64, 64), (1, 4, 96, 96, 90), (5, 3, 1, 401, 403), (2, 2, 100, 100, 97),
          (1, 3, 130, 130, 130), (3, 2, 120, 130, 130), (5, 2, 90, 95, 100)]
DOUBLES = [(3, 1, 50, 50, 50), (3, 2, 50, 50, 50), (3, 3, 50, 50, 50), (2, 4, 96, 58, 44), (4, 2, 1, 361, 363), (2, 2, 64, 64, 65),
           (1, 3, 90, 91, 92), (5, 1, 70, 70, 60)]


@pytest.mark.parametrize("shape", FLOATS)
def test_floats(shape):
    p = floats._Problem(*shape)
    floats._close(p.run("once"), p.run("local_strided"))


@pytest.mark.parametrize("shape", DOUBLES)
def test_doubles(shape):
    p = doubles._Problem(*shape)
    doubles._same(p.run("once"), p.run("local_strided"))
