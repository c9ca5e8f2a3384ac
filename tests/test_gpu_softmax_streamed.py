"""Channel softmax of tensors that are streamed past the caches (24 MiB and more, whole vectors a row) and
just below: against softmax in float64.  The bound: each output is a handful of roundings from its inputs, and
the sum over C classes of positive terms (or C products, measured in their magnitudes) one rounding a term at
most."""
import pytest

pytestmark = pytest.mark.gpu

# N, C, H, W; streamed by the larger one of a pair
CASES = [(6, 8, 362, 362), (6, 8, 364, 364), (4, 16, 320, 320), (4, 21, 270, 280), (3, 32, 256, 257), (3, 60, 200, 200),
         (2, 150, 150, 150), (8, 250, 60, 60), (1, 400, 130, 130), (5, 600, 48, 48)]


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("shape", CASES)
def test_streamed_softmax(shape, dtype):
    import torch
    from dihydrogen_amd.layers import Softmax, SoftmaxMode
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    tdt = getattr(torch, dtype)
    eps = torch.finfo(tdt).eps
    make = lambda: Tensor(list(shape[::-1]), LocaleVirtual(0, 1), Distribution.make_localized_distribution(4), tdt).allocate()
    x, y, dy, dx = (make() for _ in range(4))
    g = torch.Generator(device="cuda").manual_seed(shape[1])
    x.real_view().normal_(0, 2, generator=g)
    dy.real_view().normal_(0, 1, generator=g)
    sm = Softmax()
    sm.setup(x, SoftmaxMode.CHANNEL)
    assert sm.forward(x, y) == 0 and sm.backward(y, dy, dx) == 0
    torch.cuda.synchronize()
    c = shape[1]
    for n in range(shape[0]):  # a sample at a time: the reference is in float64
        want = torch.softmax(x.real_view()[n].double(), 0)
        got = y.real_view()[n].double()
        assert bool(((got - want).abs() <= (c + 16) * eps * want).all())
        d = dy.real_view()[n].double()
        dot = (got * d).sum(0)
        magnitude = got * (d.abs() + (got * d).abs().sum(0))
        assert bool(((dx.real_view()[n].double() - got * (d - dot)).abs() <= (c + 4) * eps * magnitude).all())
