"""Normalising haloed tensors with statistics that are given: outputs up to 32 MiB are stored normally but for some of one plane, larger
ones past the caches.
The samples of a larger tensor, all at once and in two halves: the same bits, and the halo as it was."""
import pytest
import torch

from dihydrogen_amd.layers import BatchNormalization
from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor

pytestmark = pytest.mark.gpu

# rows of whole vectors and not, shorter than a vector, short segments (up to 256 elements) and longer ones; N is made from the size
SHAPES = [((9, 9), 1), ((8, 12), 2), ((2, 11), 1), ((1, 30), 2), ((40, 41), 1), ((64, 64), 3), ((3, 200), 1), ((6, 7, 8), 1), ((31, 30, 29), 2)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("spatial,halo", SHAPES)
def test_all_at_once_and_in_halves(spatial, halo, dtype):
    ns, c = len(spatial), 5
    dist = Distribution.make_overlapped_distribution([2] * ns + [1, 1], [halo] * ns + [0, 0])
    make = lambda n: Tensor([2 * e for e in spatial] + [c, n], LocaleVirtual(0, 2 ** ns), dist, dtype).allocate()
    one = make(1)
    n = 2 * ((17 << 20) // (one.data.numel() * one.data.element_size()) + 1)  # halves of 17 MiB, or a sample more
    x, y = make(n), make(n)
    x.data.normal_(0, 1, generator=torch.Generator(device="cuda").manual_seed(n))
    y.data.fill_(7)
    layer = BatchNormalization(ns + 2, 0.9, 1e-5)
    g = torch.Generator(device="cuda").manual_seed(1)
    mean, var, scale, bias = (torch.empty(c, device="cuda", dtype=dtype).uniform_(0.5, 1.5, generator=g) for _ in range(4))
    layer.set_num_samples(n)
    layer.forward(x, mean, var, mean, var, scale, bias, y, False)
    layer.set_num_samples(n // 2)
    for half in range(2):
        xh, yh = make(n // 2), make(n // 2)
        xh.data.copy_(x.data.flatten().chunk(2)[half].view_as(xh.data))
        yh.data.fill_(7)
        layer.forward(xh, mean, var, mean, var, scale, bias, yh, False)
        assert torch.equal(yh.data.flatten(), y.data.flatten().chunk(2)[half])
    inside = y.interior_view()
    shape = (1, c) + (1,) * ns
    want = (x.interior_view() - mean.view(shape)) / torch.sqrt(var.view(shape) + 1e-5) * scale.view(shape) + bias.view(shape)
    # five roundings of the type, one of them in a root; what is subtracted and added is no larger than 6
    assert (inside - want).abs().max() <= 64 * torch.finfo(dtype).eps
    rest = y.data.clone()
    y.interior_view().fill_(7)
    assert (y.data == 7).all() and rest.numel() > inside.numel()
