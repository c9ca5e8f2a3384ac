"""Whole batch-norm passes over double tensors that leave the output's halo cleared: the bits of the staged calls, and zeros in every
halo cell, by one workgroup a channel, several channels a workgroup and teams."""
import pytest
import torch

from dihydrogen_amd.layers import BatchNormalization
from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor

pytestmark = pytest.mark.gpu

# N, C, spatial extents, halo, rank of a grid of two along each dimension: segments of up to 256 elements and longer ones, channels of one
# workgroup (several sizes of it) and teams; halos on some dimensions only
SHAPES = [(3, 5, (4, 6), (1, 1)), (24, 142, (6, 6), (1, 1)), (16, 47, (7, 6), (2, 2)), (9, 7, (3, 4, 5), (1, 2, 1)), (5, 3, (9, 1), (1, 1)),
          (26, 40, (22, 18), (1, 1)), (2, 5, (28, 23, 32), (1, 1, 1)), (20, 25, (11, 10, 7), (1, 1, 1)), (4, 30, (19, 30), (2, 0)),
          (4, 30, (19, 30), (0, 1)), (1, 29, (35, 30, 36), (1, 1, 1)), (2, 6, (20, 40, 33), (0, 1, 2)), (3, 2, (300, 40), (3, 3)),
          (2, 300, (17, 31), (1, 1)), (70, 130, (18, 16), (1, 1)), (4, 30, (64, 64), (0, 1))]
# of these the ones that stay in the staged calls, one by the estimate of the time and one whose halo on the outermost dimension alone leaves
# dense segments
STAGED = SHAPES[-2:]


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("n,c,spatial,halo", SHAPES)
def test_the_bits_of_the_staged_calls(n, c, spatial, halo, in_place):
    ns = len(spatial)
    dist = Distribution.make_overlapped_distribution([2] * ns + [1, 1], list(halo) + [0, 0])
    shape, rank = [2 * e for e in spatial] + [c, n], LocaleVirtual(0, 2 ** ns)
    make = lambda: Tensor(shape, rank, dist, torch.float64).allocate()
    g = torch.Generator(device="cuda").manual_seed(n * c)
    x0, dy0 = (torch.randn(make().data.numel(), device="cuda", dtype=torch.float64, generator=g) for _ in range(2))
    scale, bias = (torch.rand(c, device="cuda", dtype=torch.float64, generator=g) + 0.5 for _ in range(2))
    results = []
    for whole in (True, False):
        layer = BatchNormalization(ns + 2, 0.9, 1e-5, fuse_local=whole, clear_output_halo=True)
        x, dy, y, dx = (make() for _ in range(4))
        x.data.view(-1).copy_(x0)
        dy.data.view(-1).copy_(dy0)
        y.data.fill_(7)
        dx.data.fill_(7)
        stats = [torch.full((c,), v, device="cuda", dtype=torch.float64) for v in (0, 0, 0.25, 0.75)]
        layer.forward(x, *stats, scale, bias, y)
        grads = [torch.full((c,), 7.0, device="cuda", dtype=torch.float64) for _ in range(4)]
        into = x if in_place else dx
        layer.backward(x, dy, *stats[:2], scale, *grads, into)
        results.append([y.data.clone(), into.data.clone()] + stats + grads)
        for t in (y, into):
            t.interior_view().zero_()
            assert not t.data.any()
    for a, b in zip(*results):
        assert torch.equal(a, b)
