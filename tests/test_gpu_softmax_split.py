"""Channel softmax at the edges of the tiles whose waves share the channels, for few and for many
tiles, with one and with two pixels a lane, against float64."""
import pytest

pytestmark = pytest.mark.gpu

EDGES = [33, 64, 65, 128, 129, 192, 193, 256, 257, 384, 385, 512, 513, 768, 769, 1024, 1025]


def _check(n, c, spatial, dtype):
    import torch
    from dihydrogen_amd import capi
    lib = capi.load()
    tdt = getattr(torch, dtype)
    dt = capi.F32 if dtype == "float32" else capi.F64
    g = torch.Generator(device="cuda").manual_seed(c)
    x = torch.randn((n, c, spatial), dtype=tdt, device="cuda", generator=g) * 2
    dy = torch.randn((n, c, spatial), dtype=tdt, device="cuda", generator=g)
    guard = 64
    outs = [torch.full((x.numel() + 2 * guard,), 7, dtype=tdt, device="cuda") for _ in range(2)]
    y, dx = (o[guard:-guard].view_as(x) for o in outs)
    st = torch.cuda.current_stream().cuda_stream
    assert lib.h2x_softmax_channel_forward(dt, n, c, spatial, x.data_ptr(), y.data_ptr(), st) == 0
    assert lib.h2x_softmax_channel_backward(dt, n, c, spatial, y.data_ptr(), dy.data_ptr(), dx.data_ptr(), st) == 0
    want = torch.softmax(x.double(), 1)
    yd = y.double()
    grad = yd * (dy.double() - (yd * dy.double()).sum(1, keepdim=True))
    # exp (2 units), at most c / 4 additions in a row, a quotient and a product, a subtraction; values up to 1 and 6
    eps = torch.finfo(tdt).eps
    assert bool(((yd - want).abs() <= (8 + c / 4) * eps * want).all())
    assert bool(((dx.double() - grad).abs() <= (8 + c / 4) * eps * 6 * yd + eps * grad.abs()).all())
    for o in outs:
        assert bool((o[:guard] == 7).all()) and bool((o[-guard:] == 7).all())


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("c", EDGES)
def test_few_tiles(c, dtype):
    _check(2, c, 131, dtype)
    _check(3, c, 7, dtype)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("c", [c for c in EDGES if c <= 513])
def test_many_tiles(c, dtype):
    _check(1, c, 257 * 64 + 1, dtype)


@pytest.mark.parametrize("c", [33, 64, 65, 129, 193, 256])
def test_two_pixels_a_lane(c):
    _check(2, c, 257 * 128 + 2, "float32")
