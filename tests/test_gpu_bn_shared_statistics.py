"""Batch-norm of a program that keeps no running statistics and gives the call its buffers of the batch's mean and variance (or one
buffer of its own) for them too: what the staged calls leave there, by every way in which a whole pass runs."""
import pytest
import torch

from dihydrogen_amd.layers import BatchNormalization
from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor

pytestmark = pytest.mark.gpu

# N, C, spatial extents, halo: one workgroup a channel, windows of two channels, a team, two launches; of doubles short segments,
# one workgroup, a team
SHAPES = [(torch.float32, 8, 5, (32, 32), 0), (torch.float32, 128, 1023, (7, 7), 0), (torch.float32, 2, 3, (40, 32, 32), 0),
          (torch.float32, 3, 7, (2, 1), 0), (torch.float32, 2, 96, (61, 32), 2), (torch.float64, 30, 70, (10, 11), 0),
          (torch.float64, 3, 3, (45, 47), 0), (torch.float64, 2, 2, (32, 32, 40), 0), (torch.float64, 60, 20, (6, 4), 1)]
KERNELS = [[8], [9], [10], [0, 1], [8], [13], [11], [12], [13]]  # forward, of each: see h2x_bn_planned


@pytest.mark.parametrize("one_buffer", [False, True])
@pytest.mark.parametrize("clear", [False, True])
@pytest.mark.parametrize("dtype,n,c,spatial,halo", SHAPES)
def test_as_in_the_staged_calls(dtype, n, c, spatial, halo, clear, one_buffer):
    ns = len(spatial)
    dist = Distribution.make_overlapped_distribution([2] * ns + [1, 1], [halo] * ns + [0, 0])
    make = lambda: Tensor([2 * e for e in spatial] + [c, n], LocaleVirtual(0, 2 ** ns), dist, dtype).allocate()
    g = torch.Generator(device="cuda").manual_seed(n * c)
    x, dy = make(), make()
    x.data.normal_(1, 2, generator=g)
    dy.data.normal_(0, 1, generator=g)
    scale, bias = (torch.empty(c, device="cuda", dtype=dtype).uniform_(0.5, 1.5, generator=g) for _ in range(2))
    results = []
    for whole in (True, False):
        layer = BatchNormalization(ns + 2, 0.9, 1e-5, fuse_local=whole, clear_output_halo=clear)
        y, dx = make(), make()
        mean, var, spare = (torch.full((c,), v, device="cuda", dtype=dtype) for v in (0, 0, 0.25))
        running = (spare, spare) if one_buffer else (mean, var)
        layer.forward(x, mean, var, *running, scale, bias, y)
        grads = [torch.empty(c, device="cuda", dtype=dtype) for _ in range(4)]
        layer.backward(x, dy, mean, var, scale, *grads, dx)
        results.append([y.interior_view(), dx.interior_view(), mean, var, spare] + grads)
    for a, b in zip(*results):
        # the order of the fp64 sums: 16 units in the last place of the largest value, as of separate buffers; of what is left in the
        # buffers of the statistics, two roundings more
        assert ((a - b).abs() <= 18 * torch.finfo(dtype).eps * b.abs().max()).all()
