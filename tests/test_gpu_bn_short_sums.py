"""Batch-norm of doubles in short segments in one launch, whose sums of rows of lanes and of ranges are read eight at a time: numbers of
samples at which a batch of either is just full or not, against the two-launch calls, bit for bit."""
import pytest

import test_gpu_bn_ordered as ordered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("segment", [(1, 1), (1, 2), (2, 3), (5, 5), (13, 13)])
@pytest.mark.parametrize("n", [2, 8, 9, 10, 16, 17, 18, 31, 33, 34, 65, 66, 129, 145, 250])
def test_the_bits_of_two_launches(n, segment):
    p = ordered._Problem(n, 45, 1, *segment, 0)
    ordered._same(p.run("once"), p.run("local_strided"))
