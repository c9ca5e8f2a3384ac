"""Batch-norm with channels held in registers, by one workgroup or by a team, against the two-launch
calls, at the edges of the variants (vectors a channel: the tile sizes and one more)."""
import ctypes

import pytest

from dihydrogen_amd import capi

pytestmark = pytest.mark.gpu


class _Problem:
    """One haloed (or dense) N, C, D, H, W tensor set and the three ways to run it."""

    def __init__(self, n, c, d, h, w, halo=0):
        import torch
        self.torch, self.n, self.c = torch, n, c
        hd = halo if d > 1 else 0
        real = (n, c, d + 2 * hd, h + 2 * halo, w + 2 * halo)
        g = torch.Generator(device="cuda").manual_seed(n + c + w)
        self.x, self.dy = (torch.randn(real, device="cuda", generator=g) for _ in range(2))
        self.x += 0.5
        self.inner = (slice(None), slice(None), slice(hd, hd + d), slice(halo, halo + h), slice(halo, halo + w))
        first = hd * self.x.stride(2) + halo * self.x.stride(3) + halo
        self.offset = first * self.x.element_size()
        self.geometry = capi.TensorGeometry()
        self.geometry.num_dims = 5
        for i, (e, s) in enumerate(zip((w, h, d, c, n), reversed(self.x.stride()))):
            self.geometry.local_shape[i], self.geometry.strides[i] = e, s
        self.per = n * d * h * w
        self.scale = torch.empty(c, device="cuda").uniform_(0.5, 1.5, generator=g)
        self.bias = torch.empty(c, device="cuda").normal_(0, 0.1, generator=g)
        self.ws = torch.empty(capi.load().h2x_bn_workspace_bytes(c), dtype=torch.uint8, device="cuda")
        self.state = torch.zeros(capi.load().h2x_bn_team_state_bytes(c), dtype=torch.uint8, device="cuda")

    def run(self, kind, *polls, in_place=False):
        """(outputs, halo untouched?) of h2x_bn_{forward,backward}_<kind>."""
        torch, lib = self.torch, capi.load()
        gp = ctypes.byref(self.geometry)
        vec = lambda v: torch.full_like(self.scale, v)
        mean, var, rm, rv = vec(float("nan")), vec(float("nan")), vec(0.25), vec(0.75)
        grads = [vec(float("nan")) for _ in range(4)]
        x = self.x.clone()
        y = x if in_place else torch.full_like(x, 7)
        at = lambda t: t.data_ptr() + self.offset
        p = lambda t: t.data_ptr()
        st = torch.cuda.current_stream().cuda_stream
        scratch = {"once": [p(self.ws), p(self.state)], "team": [p(self.state)]}.get(kind, [p(self.ws)])
        status = getattr(lib, "h2x_bn_forward_" + kind)(
            capi.F32, self.n, gp, gp, at(x), p(self.scale), p(self.bias), self.per, 0.9, 1e-5, p(mean), p(var), p(rm),
            p(rv), at(y), *scratch, *polls, st)
        assert status == 0, status
        if in_place:
            x = self.x.clone()
        dx = x if in_place else torch.full_like(x, 7)
        status = getattr(lib, "h2x_bn_backward_" + kind)(
            capi.F32, self.n, self.per, gp, gp, gp, at(x), at(self.dy), p(mean), p(var), p(self.scale),
            *[p(t) for t in grads], at(dx), 1e-5, *scratch, *polls, st)
        assert status == 0, status
        torch.cuda.synchronize()
        for out in (y, dx):
            if not in_place:
                rest = out.clone()
                rest[self.inner] = 7
                assert bool((rest == 7).all()), "stored outside the interior"
        return [y[self.inner], dx[self.inner], mean, var, rm, rv] + grads


def _close(got, want):
    """The fp64 sums differ by their order only (2^-52 of the sum of the terms' magnitudes), so the statistics by at
    most a rounding to float; a handful of operations follow: 16 units in the last place of the
    largest value."""
    for a, b in zip(got, want):
        assert bool(((a - b).abs() <= 16 * 1.2e-7 * b.abs().max()).all())


# vectors a channel of the variants' edges; 96 channels reach the largest ones
ONCE = [(1, 5, 1, 16, 32), (1, 5, 1, 3, 172), (2, 3, 1, 32, 64), (3, 3, 1, 37, 37), (8, 3, 1, 32, 32),
        (8, 3, 1, 32, 64), (5, 2, 1, 59, 111), (4, 97, 1, 128, 128), (4, 96, 1, 128, 129), (5, 96, 1, 128, 128),
        (40, 1030, 1, 7, 7), (3, 7, 1, 2, 2), (4, 96, 1, 64, 65), (4, 65, 1, 64, 64), (9, 43, 1, 43, 44)]


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("shape", ONCE)
def test_channel_in_one_workgroup(shape, in_place):
    p = _Problem(*shape)
    _close(p.run("once", in_place=in_place), p.run("local_strided"))


@pytest.mark.parametrize("shape", [(2, 5, 6, 9, 11), (4, 70, 4, 5, 30), (2, 96, 16, 32, 61)])
def test_haloed_channel_in_one_workgroup(shape):
    p = _Problem(*shape, halo=2)
    _close(p.run("once"), p.run("local_strided"))


# few members and many, a last member that is nearly empty, haloed rows; the last three
# reach every variant and both kinds of stores by the dispatch's own rule
TEAM = [(1, 3, 1, 64, 300, 0), (2, 2, 40, 32, 32, 0), (1, 2, 33, 35, 37, 1),
        (3, 2, 1, 257, 129, 0), (2, 3, 17, 18, 19, 2), (31, 2, 64, 32, 32, 0),
        (2, 32, 48, 48, 48, 0), (5, 24, 48, 48, 48, 0), (2, 64, 45, 62, 62, 1)]


@pytest.mark.parametrize("shape", TEAM)
def test_channel_in_a_team(shape):
    """As the two-launch calls, and with the same bits when no member waits and each works out
    the sums of all others."""
    import torch
    p = _Problem(*shape)
    by_team = p.run("team", 2048)
    _close(by_team, p.run("local_strided"))
    small = p.x.numel() < 4_000_000  # every member reads its whole channel
    for polls in ([0, 2048] if small else [2048, 2048]):  # and again with the state that these calls leave
        for a, b in zip(by_team, p.run("team", polls)):
            assert torch.equal(a, b)
    _close(p.run("once"), by_team)


# 33 to 64 members a channel: two waves look after them forward, three and four backward
@pytest.mark.parametrize("shape", [(1, 1, 1, 800, 820, 0), (1, 2, 62, 90, 94, 1), (1, 1, 1, 900, 1160, 0)])
def test_members_that_several_waves_look_after(shape):
    """The same bits when all, some or none of the others' sums are worked out."""
    import torch
    p = _Problem(*shape)
    counter = p.state.view(torch.int64)[:1]
    by_team = p.run("team", 2048)
    assert int(counter) > 2 * 32    # members, forward and backward: each has added one
    _close(by_team, p.run("local_strided"))
    for polls in (0, 1, 2, 3, 2048):
        for a, b in zip(by_team, p.run("team", polls)):
            assert torch.equal(a, b)


def test_one_state_for_calls_of_other_sizes():
    """Teams of other sizes, forward and backward, leave sums of earlier calls in the state: none is taken for a new one."""
    import torch
    problems = [_Problem(*s) for s in [(2, 3, 40, 32, 32), (7, 3, 40, 32, 32), (1, 3, 1, 64, 300), (3, 2, 17, 18, 19, 2)]]
    wants = [p.run("team", 2048) for p in problems]
    state = problems[0].state
    for i in (0, 1, 2, 1, 3, 0, 2, 3, 1):
        problems[i].state = state
        for a, b in zip(problems[i].run("team", 2048), wants[i]):
            assert torch.equal(a, b)


def test_nan_reaches_the_whole_channel_of_a_team_only():
    import torch
    p = _Problem(2, 3, 40, 32, 32)
    p.x[1, 1, 30, 2, 3] = float("nan")
    out, ref = p.run("team", 2048), p.run("local_strided")
    for a, b in zip(out, ref):
        assert torch.equal(torch.isnan(a), torch.isnan(b))


def test_overlapping_outputs_are_not_for_teams():
    p = _Problem(2, 2, 40, 32, 32)
    x, lib, gp = p.x.data_ptr(), capi.load(), ctypes.byref(p.geometry)
    v = [p.scale.clone().data_ptr() for _ in range(4)]
    assert lib.h2x_bn_forward_team(capi.F32, 2, gp, gp, x, p.scale.data_ptr(), p.bias.data_ptr(), p.per, 0.9, 1e-5, *v, x,
                                   p.state.data_ptr(), 2048, None) == -2  # unsupported
    _close(p.run("once", in_place=True), p.run("local_strided"))


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("shape,halo", [((1, 2, 5, 6, 6), 1), ((3, 5, 10, 10, 10), 1), ((4, 3, 1, 30, 30), 1),
                                        ((2, 4, 1, 58, 30), 3), ((2, 100, 30, 30, 30), 1), ((16, 64, 30, 30, 30), 1),
                                        ((2, 64, 44, 62, 62), 1)])
def test_whole_pass_that_clears_the_halo(shape, halo, in_place):
    """As the two-launch calls on the interior, zeros in the halo, in one workgroup a channel and in teams
    (which outputs that overlap inputs are not for: the call refuses or is done by one workgroup)."""
    import torch
    p = _Problem(*shape, halo=halo)
    want = p.run("local_strided")
    n, c, d, h, w = shape
    hd = halo if d > 1 else 0
    g = capi.HaloedGeometry()
    g.num_dims = 5
    for i, (e, o) in enumerate(zip((w, h, d, c, n), (halo, halo, hd, 0, 0))):
        g.local_shape[i], g.real_shape[i], g.lower_halo[i] = e, e + 2 * o, o
    lib, gp = capi.load(), ctypes.byref(g)
    x, dy = (torch.full_like(t, float("nan")) for t in (p.x, p.dy))
    x[p.inner], dy[p.inner] = p.x[p.inner], p.dy[p.inner]
    vec = lambda v: torch.full_like(p.scale, v)
    mean, var, rm, rv = vec(float("nan")), vec(float("nan")), vec(0.25), vec(0.75)
    grads = [vec(float("nan")) for _ in range(4)]
    a = lambda t: t.data_ptr()
    y = x.clone() if in_place else torch.full_like(x, 7)
    status = lib.h2x_bn_forward_clearing(capi.F32, gp, a(y if in_place else x), a(p.scale), a(p.bias), p.per, 0.9, 1e-5, a(mean),
                                         a(var), a(rm), a(rv), a(y), a(p.state), None)
    if status == -2:
        assert in_place and p.x[0, 0].numel() * n > 32768
        return
    assert status == 0
    dx = x.clone() if in_place else torch.full_like(x, 7)
    assert lib.h2x_bn_backward_clearing(capi.F32, p.per, gp, a(dx if in_place else x), a(dy), a(mean), a(var), a(p.scale),
                                        *[a(t) for t in grads], a(dx), 1e-5, a(p.state), None) == 0
    torch.cuda.synchronize()
    for out in (y, dx):
        rest = out.clone()
        rest[p.inner] = 0
        assert bool((rest == 0).all())
    _close([y[p.inner], dx[p.inner], mean, var, rm, rv] + grads, want)
