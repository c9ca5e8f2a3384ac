"""Channel softmax of more channels than a lane holds: infinities, masks of the type's lowest value and NaN at the channel counts
where a register tile ends or begins, in few and in many tiles."""
import pytest
import torch

from dihydrogen_amd.layers import Softmax, SoftmaxMode
from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor

pytestmark = pytest.mark.gpu

CHANNELS = [33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 384, 385, 448, 449, 512, 513, 768, 769, 1024]
# 128 pixels counted through the samples; 5 tiles of 64 a sample; 267 and 546 tiles, odd and even rows
SHAPES = [(2, 8, 8), (3, 17, 17), (1, 130, 131), (2, 132, 132)]


def _tensor(n, c, h, w, dtype):
    return Tensor([w, h, c, n], LocaleVirtual(0, 1), Distribution.make_localized_distribution(4), dtype).allocate()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,h,w", SHAPES)
@pytest.mark.parametrize("c", CHANNELS)
def test_special_values(c, n, h, w, dtype):
    info = torch.finfo(dtype)
    x, y, dy, dx = (_tensor(n, c, h, w, dtype) for _ in range(4))
    g = torch.Generator(device="cuda").manual_seed(c * h)
    x.data.normal_(0, 2, generator=g)
    dy.data.normal_(0, 1, generator=g)
    v = x.data.view(n, c, h, w)
    v[:, 1::3, 0, :] = info.min          # masked channels
    v[:, 2::5, 1, :] = -float("inf")
    v[0, c - 1, h - 1, w - 1] = float("nan")
    v[0, 0, h - 1, w - 2] = float("inf")
    layer = Softmax()
    layer.setup(x, SoftmaxMode.CHANNEL)
    layer.forward(x, y)
    layer.backward(y, dy, dx)
    exact = torch.softmax(v.double(), 1)
    # the last pixel holds a NaN, the one before it an infinity: no number comes of either, and all is the lower bound
    exact[0, :, h - 1, w - 2:] = info.tiny
    # relative to the largest of a pixel: an exponential of an error of half a unit in x - max, and c additions
    bound = (16 + c / 8) * info.eps
    assert ((y.data.view_as(v).double() - exact).abs() <= bound * exact + 2 * info.tiny).all()
    assert (y.data >= info.tiny).all()
    yv, gv = y.data.view_as(v).double(), dy.data.view_as(v).double()
    want = torch.where(yv > info.tiny, yv * (gv - (yv * gv).sum(1, keepdim=True)), torch.zeros_like(yv))
    size = yv * (gv.abs() + (yv * gv).abs().sum(1, keepdim=True))
    assert ((dx.data.view_as(v).double() - want).abs() <= (4 + c / 8) * info.eps * size + 2 * info.tiny).all()
