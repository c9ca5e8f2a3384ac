"""Instance softmax by teams of workgroups: the bits of the staged calls, also of members that work out what they
miss, call after call on one state, and by the separate launches where a team is not for it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# samples, elements of a sample: one more than a workgroup holds; whole and single-element vectors; 64 and 65 chunks
# (members of one and of four), chunks of 4, 8 and 16 vectors a thread at their limits, and beyond (no team)
CASES = [(1, 32769), (3, 32772), (2, 64 * 4096), (2, 64 * 4096 + 4), (1, 256 * 4096), (1, 256 * 4096 + 4), (2, 256 * 8192 - 4),
         (2, 256 * 8192 + 8), (3, 256 * 8192), (3, 256 * 16384), (3, 256 * 16384 + 4), (5, 256 * 1024 - 1), (4, 256 * 2048 + 1),
         (1, 773145), (3, 1048577 * 3), (40, 51 * 4096), (70, 64 * 4096 - 4), (9, 40001)]


@pytest.mark.parametrize("polls", [-1, 0])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,size", CASES)
def test_teams_equal_the_staged_calls(n, size, dtype, polls):
    import torch
    from dihydrogen_amd import capi
    lib = capi.load()
    tdt, dt = (torch.float32, capi.F32) if dtype == np.float32 else (torch.float64, capi.F64)
    g = torch.Generator(device="cuda").manual_seed(size)
    need = lib.h2x_softmax_instance_state_needed(dt, n, size)
    assert (need > 0) == (size * np.dtype(dtype).itemsize <= 256 * 16384 * {1: 1, 2: 2}.get(n, 4))
    state = torch.zeros(max(need, 8), dtype=torch.uint8, device="cuda")
    ws = torch.empty(lib.h2x_softmax_instance_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    p = lambda t: t.data_ptr()
    per_sample = lambda: torch.full((n,), float("nan"), device="cuda", dtype=tdt)
    for call in range(3):
        x = torch.randn(n, size, device="cuda", dtype=tdt, generator=g) * 2
        dy = torch.randn(n, size, device="cuda", dtype=tdt, generator=g)
        if call == 1:
            x[0, 5], x[-1, -1] = (float("inf") if n > 1 else 90.0), float("nan")
        outs = []
        for team in (True, False):
            mx, ex, dp = per_sample(), per_sample(), per_sample()
            y, dx = torch.full_like(x, 7), torch.full_like(x, 7)
            if team:
                in_place = call == 2
                a, d = (x.clone(), dy.clone()) if in_place else (x, dy)
                y, dx = (a, d) if in_place else (y, dx)
                capi.check(lib.h2x_softmax_instance_forward_once(dt, n, size, p(a), p(y), p(mx), p(ex), p(ws), p(state), polls, None))
                capi.check(lib.h2x_softmax_instance_backward_once(dt, n, size, p(y), p(d), p(dx), p(dp), p(ws), p(state), polls,
                                                                  None))
            else:
                capi.check(lib.h2x_softmax_instance_max(dt, n, size, p(x), p(mx), p(ws), None))
                capi.check(lib.h2x_softmax_instance_exp(dt, n, size, p(x), p(mx), p(y), p(ex), p(ws), None))
                capi.check(lib.h2x_softmax_instance_normalize(dt, n, size, p(ex), p(y), None))
                capi.check(lib.h2x_softmax_instance_dot(dt, n, size, p(y), p(dy), p(dp), p(ws), None))
                capi.check(lib.h2x_softmax_instance_gradient(dt, n, size, p(y), p(dy), p(dp), p(dx), None))
            torch.cuda.synchronize()
            outs.append((mx, ex, y, dp, dx))
        for name, a, b in zip(("max", "sum", "y", "dot", "dx"), *outs):
            same = (a == b) | (torch.isnan(a) & torch.isnan(b))
            assert bool(same.all()), (name, call)
    if need:
        # one arrival a member and direction: in place there is no team
        members = state.view(torch.int64)[: need // 8].reshape(n, -1)[:, 0] // 4
        assert bool((members > 1).all()) and bool((members <= 256).all())


def test_layer_calls_on_growing_batches():
    """One layer, tensors of different batch and sample sizes: against softmax in float64."""
    import torch
    from dihydrogen_amd.layers import Softmax, SoftmaxMode
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    sm = Softmax()
    for n, c, h, w in ((2, 9, 70, 71), (5, 16, 64, 64), (1, 81, 115, 83), (5, 16, 64, 64)):
        make = lambda: Tensor([w, h, c, n], LocaleVirtual(0, 1), Distribution.make_localized_distribution(4),
                              torch.float32).allocate()
        x, y, dy, dx = (make() for _ in range(4))
        x.real_view().normal_(0, 2), dy.real_view().normal_(0, 1)
        sm.setup(x, SoftmaxMode.INSTANCE)
        assert sm.forward(x, y) == 0 and sm.backward(y, dy, dx) == 0
        torch.cuda.synchronize()
        flat = lambda t: t.real_view().reshape(n, -1).double()
        want, got, d = torch.softmax(flat(x), 1), flat(y), flat(dy)
        eps = torch.finfo(torch.float32).eps
        assert bool(((got - want).abs() <= 16 * eps * want).all())
        dot = (got * d).sum(1, keepdim=True)
        # three roundings and that of the dot product, whose terms are added in float64
        assert bool(((flat(dx) - got * (d - dot)).abs() <= 4 * eps * got * (d.abs() + dot.abs())).all())


@pytest.mark.parametrize("before", [False, True])
def test_replayed_calls(before):
    """Calls in a captured graph, the state made before or during the capture, with calls on it in between."""
    import torch
    from dihydrogen_amd.layers import Softmax, SoftmaxMode
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    make = lambda: Tensor([64, 64, 30, 2], LocaleVirtual(0, 1), Distribution.make_localized_distribution(4),
                          torch.float32).allocate()
    x, y, dy, dx = (make() for _ in range(4))
    layers = [Softmax() for _ in range(2)]
    for sm in layers:
        sm.setup(x, SoftmaxMode.INSTANCE)
    run = lambda sm: (sm.forward(x, y), sm.backward(y, dy, dx))
    run(layers[1])
    if before:
        run(layers[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(layers[0])
    for replay in range(4):
        x.data.normal_(0, 2), dy.data.normal_(0, 1)
        run(layers[replay % 2])
        torch.cuda.synchronize()
        want = y.data.clone(), dx.data.clone()
        y.data.fill_(7), dx.data.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.data, want[0]) and torch.equal(dx.data, want[1])


def test_size_of_the_state():
    """Two partials of up to 64 members a sample, and a line."""
    from dihydrogen_amd import capi
    need = capi.load().h2x_softmax_instance_state_needed
    for dtype in (capi.F32, capi.F64):
        for n, size in ((1, 40001), (3, 64 * 4096), (2, 256 * 2048), (40, 51 * 4096)):
            assert need(dtype, n, size) == n * (128 + 2 * 64 * 2 * 8)


# samples of single elements around 64 chunks, and of chunks around 32 KB, whose members are one round of the chip or two
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,size", [(2, 64 * 4096 - 1), (2, 64 * 4096 + 1), (3, 256 * 8192 - 1), (4, 256 * 8192 + 1)])
def test_samples_of_single_elements(n, size, dtype):
    test_teams_equal_the_staged_calls(n, size, dtype, -1)


@pytest.mark.parametrize("n,size,team", [(5, 3054213, False), (3, 2097657, False), (3, 3145731, True),
                                         (5, 1596595, True), (5, 3063970, False), (4, 3932156, True)])
def test_large_chunks_of_single_elements(n, size, team):
    from dihydrogen_amd import capi
    assert (capi.load().h2x_softmax_instance_state_needed(capi.F32, n, size) > 0) == team


# members of 256 KB on three quarters of the chip, of 128 KB on a little more than all of it; members of 256 KB on 240 CUs
@pytest.mark.parametrize("n,size,team", [(6, 2145024, False), (7, 1280796, False), (4, 3932160, True), (256, 40001, True)])
def test_forward_by_teams_where_it_pays(n, size, team):
    """A member counts its arrival in the state of its sample."""
    import torch
    from dihydrogen_amd import capi
    lib, p = capi.load(), lambda t: t.data_ptr()
    x = torch.randn(n, size, device="cuda")
    y, mx, ex = torch.empty_like(x), torch.empty(n, device="cuda"), torch.empty(n, device="cuda")
    ws = torch.empty(lib.h2x_softmax_instance_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    state = torch.zeros(lib.h2x_softmax_instance_state_needed(capi.F32, n, size) + 8, dtype=torch.uint8, device="cuda")
    capi.check(lib.h2x_softmax_instance_forward_once(capi.F32, n, size, p(x), p(y), p(mx), p(ex), p(ws), p(state), -1, None))
    torch.cuda.synchronize()
    assert bool(state.any()) == team


# members of one chunk and of four, whose vectors are whole or single elements by the alignment of what takes part in the cut
@pytest.mark.parametrize("team", [True, False])
@pytest.mark.parametrize("skewed", ["x", "y", "dy", "dx"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,size", [(3, 32772), (2, 64 * 4096), (2, 64 * 4096 + 4), (3, 256 * 4096)])  # within a backward team
def test_one_tensor_off_alignment(n, size, dtype, skewed, team):
    """The staged calls' bits, by teams and by the separate launches.  dx takes no part in the cut: beside aligned y and dy
    no team serves it."""
    import torch
    from dihydrogen_amd import capi
    lib, p = capi.load(), lambda t: t.data_ptr()
    tdt, dt = (torch.float32, capi.F32) if dtype == np.float32 else (torch.float64, capi.F64)
    room = {name: torch.full((n * size + 2,), 7.0, device="cuda", dtype=tdt) for name in ("x", "y", "dy", "dx", "ys", "dxs")}
    t = {name: r[int(name.rstrip("s") == skewed):][:n * size].view(n, size) for name, r in room.items()}
    t["x"].normal_(0, 2), t["dy"].normal_(0, 1)
    ws = torch.empty(lib.h2x_softmax_instance_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    state = torch.zeros(lib.h2x_softmax_instance_state_needed(dt, n, 40001), dtype=torch.uint8, device="cuda")
    mx, ex, dp, mxs, exs, dps = (torch.empty(n, device="cuda", dtype=tdt) for _ in range(6))
    at = p(state) if team else None
    capi.check(lib.h2x_softmax_instance_forward_once(dt, n, size, p(t["x"]), p(t["y"]), p(mx), p(ex), p(ws), at, -1, None))
    torch.cuda.synchronize()
    arrivals = state.view(torch.int64).reshape(n, -1)[:, 0].clone()
    capi.check(lib.h2x_softmax_instance_backward_once(dt, n, size, p(t["y"]), p(t["dy"]), p(t["dx"]), p(dp), p(ws), at, -1, None))
    capi.check(lib.h2x_softmax_instance_max(dt, n, size, p(t["x"]), p(mxs), p(ws), None))
    capi.check(lib.h2x_softmax_instance_exp(dt, n, size, p(t["x"]), p(mxs), p(t["ys"]), p(exs), p(ws), None))
    capi.check(lib.h2x_softmax_instance_normalize(dt, n, size, p(exs), p(t["ys"]), None))
    capi.check(lib.h2x_softmax_instance_dot(dt, n, size, p(t["ys"]), p(t["dy"]), p(dps), p(ws), None))
    capi.check(lib.h2x_softmax_instance_gradient(dt, n, size, p(t["ys"]), p(t["dy"]), p(dps), p(t["dxs"]), None))
    torch.cuda.synchronize()
    served = state.view(torch.int64).reshape(n, -1)[:, 0] > arrivals
    assert bool(served.any()) == (team and skewed != "dx") and bool(served.all()) == bool(served.any())
    for a, b in ((mx, mxs), (ex, exs), (t["y"], t["ys"]), (dp, dps), (t["dx"], t["dxs"])):
        assert torch.equal(a, b)
    for name, r in room.items():  # nothing beside the tensors was written
        first = int(name.rstrip("s") == skewed)
        assert bool((r[:first] == 7).all()) and bool((r[first + n * size:] == 7).all())


# members of four chunks of 8 KB, of few samples; of one of 16 KB; whole vectors, members of four in two rounds of the chip
@pytest.mark.parametrize("n,size,members", [(2, 439890, 54), (3, 332793, 41), (12, 241997, 60), (7, 1004304, 62)])
def test_members_of_a_forward_pass(n, size, members):
    import torch
    from dihydrogen_amd import capi
    lib, p = capi.load(), lambda t: t.data_ptr()
    x = torch.randn(n, size, device="cuda")
    y, mx, ex = torch.empty_like(x), torch.empty(n, device="cuda"), torch.empty(n, device="cuda")
    ws = torch.empty(lib.h2x_softmax_instance_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    state = torch.zeros(lib.h2x_softmax_instance_state_needed(capi.F32, n, 40001), dtype=torch.uint8, device="cuda")
    capi.check(lib.h2x_softmax_instance_forward_once(capi.F32, n, size, p(x), p(y), p(mx), p(ex), p(ws), p(state), -1, None))
    torch.cuda.synchronize()
    arrivals = state.view(torch.int64).reshape(n, -1)[:, 0]
    assert arrivals.tolist() == [members] * n
    assert bool(((y.double() - torch.softmax(x.double(), 1)).abs() <= 16 * torch.finfo(torch.float32).eps * y.double()).all())
