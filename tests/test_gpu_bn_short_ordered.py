"""Batch-norm of double tensors of short segments that reads every element once: the bits of the two-launch calls."""
import pytest

import test_gpu_bn_ordered as ordered

pytestmark = pytest.mark.gpu

# one and several ranges of samples, rows of lanes, ranges one after another in a lane; the smallest and the longest segments, rows of one
# element, of one vector and of one more, with a halo and without; channels that do not fill a last window; every size of workgroup
SHAPES = [(2, 1, 1, 1, 1, 0), (33, 70, 1, 1, 1, 0), (256, 700, 1, 1, 1, 0), (200, 70, 1, 3, 1, 1), (12, 300, 1, 1, 2, 0),
          (17, 4, 1, 9, 1, 1), (3, 11, 2, 3, 5, 1), (7, 9, 3, 5, 7, 2), (9, 5, 1, 7, 7, 0), (1, 1000, 1, 2, 2, 0),
          (40, 3, 4, 4, 4, 1), (100, 37, 1, 5, 5, 0), (222, 33, 1, 4, 4, 0), (60, 200, 1, 4, 6, 1), (30, 70, 1, 10, 11, 0),
          (30, 3, 1, 16, 16, 0), (50, 275, 1, 18, 9, 2), (120, 276, 1, 9, 14, 0), (109, 1100, 1, 5, 6, 0), (128, 512, 1, 7, 7, 0),
          (64, 2, 1, 17, 15, 0), (24, 64, 1, 14, 13, 1), (26, 64, 1, 12, 14, 0), (126, 66, 1, 14, 6, 0),
          (24, 1, 1, 12, 12, 0), (194, 6, 1, 5, 1, 1)]


@pytest.mark.parametrize("shape", SHAPES)
def test_the_bits_of_two_launches(shape):
    p = ordered._Problem(*shape)
    ordered._same(p.run("once"), p.run("local_strided"))


@pytest.mark.parametrize("shape", SHAPES)
def test_in_place(shape):
    """The same interior; the halo is the input's."""
    p = ordered._Problem(*shape)
    want = p.run("local_strided")
    for i in range(2):
        whole = p.x.clone()
        whole[p.inner] = want[i][p.inner]
        want[i] = whole
    ordered._same(p.run("once", in_place=True), want)


def test_tensors_off_a_vector_boundary():
    p = ordered._Problem(30, 41, 1, 5, 7, skew=1)
    ordered._same(p.run("once"), p.run("local_strided"))


def test_special_values_stay_in_their_channel():
    p = ordered._Problem(20, 40, 1, 3, 5)
    p.x[3, 7, 0, 2, 4] = float("nan")  # the last element of a channel, side by side with the next one's first
    p.dy[5, 21, 0, 0, 0] = float("inf")
    p.x[:, 30] = 1e-200                # squares below the smallest number
    ordered._same(p.run("once"), p.run("local_strided"))
