"""Instance softmax of samples beyond one workgroup: the passes that combine the partials of the reduction
before them give the bits of the staged calls, which launch a kernel to do so.  At the edges: one more element
than a workgroup holds, as many partials as a workgroup combines (256) and one more, as many as the
workspace holds for both reductions and more, odd sizes, in place."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# samples, elements of a sample
CASES = [(1, 32769), (3, 158652), (2, 256 * 4096), (2, 256 * 4096 + 4), (1, 256 * 1024 - 1), (1, 256 * 1024 + 1),
         (40, 51 * 4096), (40, 52 * 4096), (9, 40001)]


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,size", CASES)
def test_whole_passes_equal_the_staged_calls(n, size, dtype, in_place):
    import torch
    from dihydrogen_amd import capi
    lib = capi.load()
    tdt, dt = (torch.float32, capi.F32) if dtype == np.float32 else (torch.float64, capi.F64)
    g = torch.Generator(device="cuda").manual_seed(size)
    x = torch.randn(n, size, device="cuda", dtype=tdt, generator=g) * 2
    dy = torch.randn(n, size, device="cuda", dtype=tdt, generator=g)
    x[0, 5] = float("inf") if n > 1 else 90.0
    ws = torch.empty(lib.h2x_softmax_instance_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    p = lambda t: t.data_ptr()
    per_sample = lambda: torch.full((n,), float("nan"), device="cuda", dtype=tdt)
    outs = []
    for local in (True, False):
        mx, ex, dp = per_sample(), per_sample(), per_sample()
        a = x.clone()
        y = a if in_place and local else torch.full_like(x, 7)
        if local:
            capi.check(lib.h2x_softmax_instance_forward_local(dt, n, size, p(a), p(y), p(mx), p(ex), p(ws), None))
        else:
            capi.check(lib.h2x_softmax_instance_max(dt, n, size, p(a), p(mx), p(ws), None))
            capi.check(lib.h2x_softmax_instance_exp(dt, n, size, p(a), p(mx), p(y), p(ex), p(ws), None))
            capi.check(lib.h2x_softmax_instance_normalize(dt, n, size, p(ex), p(y), None))
        d = dy.clone()
        dx = d if in_place and local else torch.full_like(x, 7)
        y_kept = y.clone()
        if local:
            capi.check(lib.h2x_softmax_instance_backward_local(dt, n, size, p(y), p(d), p(dx), p(dp), p(ws), None))
        else:
            capi.check(lib.h2x_softmax_instance_dot(dt, n, size, p(y), p(d), p(dp), p(ws), None))
            capi.check(lib.h2x_softmax_instance_gradient(dt, n, size, p(y), p(d), p(dp), p(dx), None))
        torch.cuda.synchronize()
        outs.append([t.cpu().numpy() for t in (mx, ex, y_kept, dp, dx)])
    for name, a, b in zip(("max", "sum", "y", "dot", "dx"), *outs):
        assert np.array_equal(a, b, equal_nan=True), name
