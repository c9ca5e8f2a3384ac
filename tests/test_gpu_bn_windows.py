"""Batch-norm with two or four channels of short segments in a workgroup, against the two-launch calls: an odd channel at
the end, the turns of the samples and one more, the shortest and the longest segments, memory between the channels."""
import pytest

import test_gpu_bn_once as once

pytestmark = pytest.mark.gpu

# at least 21 MiB.  Windows of two, 39 samples a turn of 7 x 7: 4 turns (full, and begun), 5, 7, 8 and 9; windows of four: 5 x 5 in 4
# turns, whole and with one, two and three channels at the end, 6 x 7
SHAPES = [(128, 1023, 1, 7, 7), (156, 701, 1, 7, 7), (157, 700, 1, 7, 7), (235, 511, 1, 7, 7), (312, 512, 1, 7, 7),
          (313, 512, 1, 7, 7), (2048, 700, 1, 2, 2), (63, 1022, 1, 1, 127), (128, 511, 1, 127, 1), (64, 1024, 1, 1, 128),
          (500, 1023, 1, 1, 11), (128, 2048, 1, 5, 5), (144, 2045, 1, 5, 5), (130, 2046, 1, 5, 5), (120, 2047, 1, 5, 5),
          (72, 1983, 1, 6, 7)]


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_two_channels_in_one_workgroup(shape, in_place):
    p = once._Problem(*shape)
    once._close(p.run("once", in_place=in_place), p.run("local_strided"))


@pytest.mark.parametrize("n,c,w,pad", [(128, 1023, 49, 2), (128, 1024, 49, 49), (128, 1024, 49, 50), (63, 1023, 127, 1),
                                       (128, 2047, 25, 3)])
def test_memory_between_the_channels(n, c, w, pad):
    """Segments that start off a vector and lie apart; what lies between them is left alone."""
    p = once._Problem(n, c, 1, 1, w + pad)
    p.inner = (Ellipsis, slice(1, 1 + w))
    p.offset, p.per, p.geometry.local_shape[0] = p.x.element_size(), n * w, w
    once._close(p.run("once"), p.run("local_strided"))


def test_nan_stays_in_its_channel():
    import torch
    p = once._Problem(128, 1024, 1, 7, 7)
    p.x[5, 10, 0, 6, 6] = float("nan")  # the last element of a channel, side by side with the next one's first
    p.dy[7, 21, 0, 0, 0] = float("inf")
    for a, b in zip(p.run("once"), p.run("local_strided")):
        assert torch.equal(torch.isnan(a), torch.isnan(b))
