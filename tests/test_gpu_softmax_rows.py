"""Softmax of samples that lanes hold in registers (instance mode, and channel mode with one pixel a
sample), at the edges of the tiles and past them, against float64."""
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 64, 65, 128, 256, 257, 512, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 16384, 16385, 32768, 32769]


def _run(kind, n, size, dtype):
    """(x, dy, y, dx) and, for instance mode, dx of the two staged calls."""
    import torch
    from dihydrogen_amd import capi
    lib = capi.load()
    tdt = getattr(torch, dtype)
    dt = capi.F32 if dtype == "float32" else capi.F64
    g = torch.Generator(device="cuda").manual_seed(size)
    x, dy = (torch.randn((n, size), dtype=tdt, device="cuda", generator=g) * 2 for _ in range(2))
    guard = 64
    outs = [torch.full((x.numel() + 2 * guard,), 7, dtype=tdt, device="cuda") for _ in range(3)]
    y, dx, staged = (o[guard:-guard].view_as(x) for o in outs)
    st = torch.cuda.current_stream().cuda_stream
    if kind == "channel":
        assert lib.h2x_softmax_channel_forward(dt, n, size, 1, x.data_ptr(), y.data_ptr(), st) == 0
        assert lib.h2x_softmax_channel_backward(dt, n, size, 1, y.data_ptr(), dy.data_ptr(), dx.data_ptr(), st) == 0
    else:
        ws = torch.empty(lib.h2x_softmax_instance_workspace_bytes(n), dtype=torch.uint8, device="cuda")
        s = torch.empty((2, n), dtype=tdt, device="cuda")
        assert lib.h2x_softmax_instance_forward_local(dt, n, size, x.data_ptr(), y.data_ptr(), s[0].data_ptr(),
                                                      s[1].data_ptr(), ws.data_ptr(), st) == 0
        assert lib.h2x_softmax_instance_backward_local(dt, n, size, y.data_ptr(), dy.data_ptr(), dx.data_ptr(),
                                                       s[0].data_ptr(), ws.data_ptr(), st) == 0
        assert lib.h2x_softmax_instance_dot(dt, n, size, y.data_ptr(), dy.data_ptr(), s[1].data_ptr(),
                                            ws.data_ptr(), st) == 0
        assert lib.h2x_softmax_instance_gradient(dt, n, size, y.data_ptr(), dy.data_ptr(), s[1].data_ptr(),
                                                 staged.data_ptr(), st) == 0
        assert torch.equal(s[0], s[1]) and torch.equal(dx, staged)
    for o in outs:
        assert bool((o[:guard] == 7).all()) and bool((o[-guard:] == 7).all())
    return x, dy, y, dx


def _check(kind, n, size, dtype):
    import torch
    x, dy, y, dx = _run(kind, n, size, dtype)
    e = torch.exp(x.double() - x.double().amax(1, keepdim=True))
    want = e / e.sum(1, keepdim=True)  # (torch.softmax of more than 1024 doubles is right to seven digits here)
    yd = y.double()
    grad = yd * (dy.double() - (yd * dy.double()).sum(1, keepdim=True))
    # exp (2 units), at most 32 + 10 additions in a row (kernels that walk a sample: size / 256), a quotient
    # and a product; dy up to about 12
    eps = torch.finfo(y.dtype).eps * (50 + size / 256)
    assert bool(((y.double() - want).abs() <= eps * want).all())
    assert bool(((dx.double() - grad).abs() <= 12 * eps * yd + eps * grad.abs()).all())


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("kind", ["instance", "channel"])
@pytest.mark.parametrize("size", SIZES)
def test_few_samples(size, kind, dtype):
    _check(kind, 5, size, dtype)


@pytest.mark.parametrize("kind", ["instance", "channel"])
@pytest.mark.parametrize("size", [s for s in SIZES if s <= 2049])
def test_more_samples_than_fill_the_chip_with_a_wave_each(size, kind):
    _check(kind, 2051, size, "float32")
