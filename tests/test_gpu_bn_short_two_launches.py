"""Batch-norm of short segments in two launches each way, whose second launch loads elements ahead of the sums and adds a sum in a thread: the bits of the
staged calls, at numbers of samples and channels where a batch of elements, the ranges of samples or a window of channels is full or not."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("in_place", [False, True])
# (1 x 1: windows of more sums than threads)
@pytest.mark.parametrize("channels,segment", [(1, 1), (300, 1), (130, 4), (70, 35), (5, 256), (29, 130)])
def test_the_bits_of_the_staged_calls(channels, segment, in_place, dtype):
    import torch
    from dihydrogen_amd import capi
    calls, dt, tdt = capi.calls(), capi.F32 if dtype == "float32" else capi.F64, getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(segment)
    c, s = channels, segment
    ws = torch.empty(capi.load().h2x_bn_workspace_bytes(c), dtype=torch.uint8, device="cuda")
    for n in (2, 9, 33, 67, 135, 242):
        x, dy = (torch.randn((n, c, s), dtype=tdt, device="cuda", generator=gen) for _ in range(2))
        x[n // 2, c - 1, s - 1] = float("nan") if n == 67 else 3
        scale, bias = (torch.rand(c, dtype=tdt, device="cuda", generator=gen) for _ in range(2))
        results = []
        for whole in (True, False):
            vec = lambda v: torch.full((c,), v, dtype=tdt, device="cuda")
            mean, var, rm, rv = vec(float("nan")), vec(float("nan")), vec(0.25), vec(0.75)
            grads = [vec(float("nan")) for _ in range(4)]
            y, xb = torch.full_like(x, 7), x.clone()
            dx = xb if in_place and whole else torch.full_like(x, 7)
            if whole:
                status = [calls.h2x_bn_forward_local(dt, n, c, s, s, s, x, scale, bias, n * s, 0.9, 1e-5, mean, var, rm, rv, y, ws, 0),
                          calls.h2x_bn_backward_local(dt, n, c, s, s, s, s, n * s, xb, dy, mean, var, scale, *grads, dx, 1e-5, ws, 0)]
            else:
                status = [calls.h2x_bn_channel_sums_and_sqsums(dt, n, c, s, s, x, mean, var, ws, 0),
                          calls.h2x_bn_sums_to_statistics(dt, c, n * s, 0.9, mean, var, rm, rv, 0),
                          calls.h2x_bn_batch_normalization(dt, n, c, s, s, s, x, mean, var, scale, bias, y, 1e-5, 0),
                          calls.h2x_bn_backprop1(dt, n, c, s, s, s, xb, dy, mean, var, scale, *grads, 1e-5, ws, 0),
                          calls.h2x_bn_backprop2(dt, n, c, s, s, s, s, n * s, xb, dy, mean, var, scale, grads[2], grads[3], dx, 1e-5, 0)]
            assert not any(status)
            results.append([y, mean, var, rm, rv, dx] + grads)
        for k, (a, b) in enumerate(zip(*results)):
            assert bool(((a == b) | (torch.isnan(a) & torch.isnan(b))).all()), (n, k)
        if n != 67 and n * s >= 64:  # (of few values the variance can be all cancellation)
            m, v = x.double().mean((0, 2)), x.double().var((0, 2))
            want = (x.double() - m[:, None]) / torch.sqrt(v[:, None] + 1e-5) * scale.double()[:, None] + bias.double()[:, None]
            # a mean below 1 and a variance of 0.5 to 2 (q / n - mean^2, q / n up to 3): five roundings relative to 1 or twice that, then six
            eps = torch.finfo(tdt).eps
            assert bool(((results[0][0].double() - want).abs() <= 32 * eps * (1 + want.abs())).all()), n


def test_sums_beyond_four_gigabytes_of_partials():
    """So many channels that a sum's place among a range's partials takes more than 32 bits in bytes (four sums of 8 bytes each from 2^27 channels on)."""
    import torch
    from dihydrogen_amd import capi
    calls, n, c = capi.calls(), 2, (1 << 27) + 300
    workspace = capi.load().h2x_bn_workspace_bytes(c)
    if torch.cuda.mem_get_info()[0] < workspace + (20 << 30):
        pytest.skip("not enough free device memory")
    gen = torch.Generator(device="cuda").manual_seed(5)
    ws = torch.empty(workspace, dtype=torch.uint8, device="cuda")
    x, dy = (torch.randn((n, c), device="cuda", generator=gen) for _ in range(2))
    mean, var, scale = (torch.rand(c, device="cuda", generator=gen) for _ in range(3))
    nan = lambda: torch.full((c,), float("nan"), device="cuda")
    dx, grads, staged = torch.full_like(x, 7), [nan() for _ in range(4)], [nan() for _ in range(4)]
    assert not calls.h2x_bn_backward_local(capi.F32, n, c, 1, 1, 1, 1, n, x, dy, mean, var, scale, *grads, dx, 1e-5, ws, 0)
    assert not calls.h2x_bn_backprop1(capi.F32, n, c, 1, 1, 1, x, dy, mean, var, scale, *staged, 1e-5, ws, 0)
    for a, b in zip(grads, staged):
        assert torch.equal(a, b)
    whole, dx = dx, torch.full_like(dx, 7)
    assert not calls.h2x_bn_backprop2(capi.F32, n, c, 1, 1, 1, 1, n, x, dy, mean, var, scale, staged[2], staged[3], dx, 1e-5, 0)
    assert torch.equal(whole, dx)
    del ws, x, dy, dx, whole, grads, staged, mean, var, scale, a, b
    torch.cuda.empty_cache()
