"""Instance softmax of samples of several chunks that a workgroup holds: by a team (few samples of more than four chunks), in one workgroup (in place, without
a state, many) and by the staged calls, the same bits; against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# elements of a sample, of floats (doubles: half as many): one chunk and the first beyond, the last of four chunks and the first of five, the last of
# five and the next, single-element remainders, all
SIZES = [4096, 4100, 16382, 16384, 16386, 16388, 20480, 20484, 24574, 28226, 32766, 32768]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("skew", ["", "dx", "dy"])
@pytest.mark.parametrize("n", [1, 3, 64, 76, 77, 128, 129])
def test_ways_to_run_few_large_samples(n, dtype, skew):
    import torch
    from dihydrogen_amd import capi
    lib = capi.load()
    tdt, dt = (torch.float32, capi.F32) if dtype == np.float32 else (torch.float64, capi.F64)
    g = torch.Generator(device="cuda").manual_seed(n)
    ws = torch.empty(lib.h2x_softmax_instance_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    p = lambda t: t.data_ptr()
    for size in SIZES:
        size = size if dtype == np.float32 else size // 2

        def buffer(name):
            flat = torch.full((n * size + 1,), 7, device="cuda", dtype=tdt)
            return (flat[1:] if name == skew else flat[:-1]).view(n, size)

        x = torch.randn(n, size, device="cuda", dtype=tdt, generator=g) * 2
        dy = buffer("dy").normal_(generator=g)
        need = lib.h2x_softmax_instance_state_needed(dt, n, size)
        if size * x.element_size() <= 64 << 10 or n > 128:
            assert need == 0
        elif n <= 64:
            assert need > 0
        state = torch.zeros(need, dtype=torch.uint8, device="cuda") if need else None
        per_sample = lambda: torch.full((n,), float("nan"), device="cuda", dtype=tdt)
        outs = []
        for way in ("staged", "once", "no looks", "local", "in place"):
            mx, ex, dp = per_sample(), per_sample(), per_sample()
            y, dx = torch.full_like(x, 7), buffer("dx")
            if way == "staged":
                capi.check(lib.h2x_softmax_instance_max(dt, n, size, p(x), p(mx), p(ws), None))
                capi.check(lib.h2x_softmax_instance_exp(dt, n, size, p(x), p(mx), p(y), p(ex), p(ws), None))
                capi.check(lib.h2x_softmax_instance_normalize(dt, n, size, p(ex), p(y), None))
                capi.check(lib.h2x_softmax_instance_dot(dt, n, size, p(y), p(dy), p(dp), p(ws), None))
                capi.check(lib.h2x_softmax_instance_gradient(dt, n, size, p(y), p(dy), p(dp), p(dx), None))
            elif way == "local":
                capi.check(lib.h2x_softmax_instance_forward_local(dt, n, size, p(x), p(y), p(mx), p(ex), p(ws), None))
                capi.check(lib.h2x_softmax_instance_backward_local(dt, n, size, p(y), p(dy), p(dx), p(dp), p(ws), None))
            else:
                a, d, looks = x, dy, 0 if way == "no looks" else -1
                if way == "in place":
                    a, d = x.clone(), buffer("dy").copy_(dy)
                    y, dx = a, d
                st = p(state) if need else None
                capi.check(lib.h2x_softmax_instance_forward_once(dt, n, size, p(a), p(y), p(mx), p(ex), p(ws), st, looks, None))
                kept = y.clone()
                capi.check(lib.h2x_softmax_instance_backward_once(dt, n, size, p(y), p(d), p(dx), p(dp), p(ws), st, looks, None))
                y = kept
            outs.append((mx, ex, y, dp, dx))
        for way in outs[1:]:
            for name, a, b in zip(("max", "sum", "y", "dot", "dx"), way, outs[0]):
                assert torch.equal(a, b), (size, name)
        mx, ex, y, dp, dx = outs[0]
        # of y: half a unit of the argument x - max, which the exponential makes a relative error, and of each of its result (2 units), the
        # sum (in 64 bits, 32768 terms) and the quotient; of dx: half a unit of the dot product, the difference and the product, and
        # of either side's sum of products, added in 64 bits, at most 45 additions in a row here
        eps = torch.finfo(tdt).eps
        below = x.double().amax(1, keepdim=True) - x.double()
        want = torch.exp(-below)
        want /= want.sum(1, keepdim=True)
        assert torch.equal(mx, x.amax(1))
        assert bool(((y.double() - want).abs() <= (eps * (below / 2 + 4) + 2e-14) * want).all())
        products = y.double() * dy.double()
        dot, terms = products.sum(1, keepdim=True), products.abs().sum(1, keepdim=True)
        grad = y.double() * (dy.double() - dot)
        assert bool(((dx.double() - grad).abs() <= y.double() * (2 * eps * (dy.double().abs() + dot.abs()) + 1e-14 * terms)).all())
