"""Batch-norm of double tensors that reads every element once, by one workgroup or by a team a channel: the
bits of the two-launch calls, at the edges of the variants (units of 2048 elements: one, as many as a
workgroup or a member plays, and one more)."""
import ctypes

import pytest

from dihydrogen_amd import capi

pytestmark = pytest.mark.gpu


class _Problem:
    """One haloed (or dense) N, C, D, H, W set of double tensors and the ways to run it."""

    def __init__(self, n, c, d, h, w, halo=0, skew=0):
        import torch
        self.torch, self.n, self.c = torch, n, c
        hd = halo if d > 1 else 0
        real = (n, c, d + 2 * hd, h + 2 * halo, w + 2 * halo)
        g = torch.Generator(device="cuda").manual_seed(n + c + w)
        make = lambda: torch.randn(real, device="cuda", dtype=torch.float64, generator=g)
        self.x, self.dy = make() + 0.5, make()
        if skew:  # off a 16-byte boundary
            self.x, self.dy = (torch.cat([t.new_zeros(1), t.flatten()])[1:].view(real) for t in (self.x, self.dy))
        self.inner = (slice(None), slice(None), slice(hd, hd + d), slice(halo, halo + h), slice(halo, halo + w))
        self.offset = (hd * self.x.stride(2) + halo * self.x.stride(3) + halo) * 8
        self.geometry = capi.TensorGeometry()
        self.geometry.num_dims = 5
        for i, (e, s) in enumerate(zip((w, h, d, c, n), reversed(self.x.stride()))):
            self.geometry.local_shape[i], self.geometry.strides[i] = e, s
        self.per = n * d * h * w
        self.scale = torch.empty(c, device="cuda", dtype=torch.float64).uniform_(0.5, 1.5, generator=g)
        self.bias = torch.empty(c, device="cuda", dtype=torch.float64).normal_(0, 0.1, generator=g)
        lib = capi.load()
        self.ws = torch.empty(lib.h2x_bn_workspace_bytes(c), dtype=torch.uint8, device="cuda")
        self.state = torch.zeros(lib.h2x_bn_team_state_bytes(c), dtype=torch.uint8, device="cuda")

    def run(self, kind, *polls, in_place=False):
        """Outputs of h2x_bn_{forward,backward}_<kind>, whole allocations."""
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
            capi.F64, self.n, gp, gp, at(x), p(self.scale), p(self.bias), self.per, 0.9, 1e-5, p(mean), p(var), p(rm),
            p(rv), at(y), *scratch, *polls, st)
        assert status == 0, status
        if in_place:
            x = self.x.clone()
        dx = x if in_place else torch.full_like(x, 7)
        status = getattr(lib, "h2x_bn_backward_" + kind)(
            capi.F64, self.n, self.per, gp, gp, gp, at(x), at(self.dy), p(mean), p(var), p(self.scale),
            *[p(t) for t in grads], at(dx), 1e-5, *scratch, *polls, st)
        assert status == 0, status
        torch.cuda.synchronize()
        return [y, dx, mean, var, rm, rv] + grads


def _same(got, want):
    import torch
    for a, b in zip(got, want):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))


# a channel in one unit and in two, four, eight, sixteen of them (and one more); odd segments, folded samples,
# haloed rows, rows of one vector and of one more, several rounds of units a group
ONCE = [(1, 5, 1, 16, 32, 0), (1, 3, 1, 64, 32, 0), (2, 3, 1, 64, 32, 0), (3, 3, 1, 45, 47, 0), (4, 3, 1, 64, 32, 0),
        (4, 3, 1, 64, 33, 0), (8, 100, 1, 64, 32, 0), (9, 100, 1, 64, 32, 0), (16, 97, 1, 64, 32, 0),
        (17, 97, 1, 64, 32, 0), (9, 2, 1, 17, 17, 0), (2, 5, 6, 9, 11, 2), (3, 2, 1, 700, 2, 1), (3, 2, 1, 400, 3, 1),
        (7, 21, 1, 31, 36, 2), (70, 600, 1, 20, 20, 0)]


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("shape", ONCE)
def test_channel_in_one_workgroup(shape, in_place):
    p = _Problem(*shape)
    _same(p.run("once", in_place=in_place), p.run("local_strided", in_place=in_place))


def test_tensors_off_a_vector_boundary():
    p = _Problem(3, 4, 1, 40, 64, skew=1)
    _same(p.run("once"), p.run("local_strided"))


# groups a channel: few, no whole number of members, the most that are added in one go; the last ones
# reach the variants by the dispatch's own rule
TEAM = [(1, 3, 1, 64, 300, 0), (2, 2, 40, 32, 32, 0), (1, 2, 33, 35, 37, 1), (3, 2, 1, 257, 129, 0),
        (2, 3, 17, 18, 19, 2), (2, 32, 48, 48, 48, 0), (8, 32, 33, 33, 33, 0), (4, 9, 1, 113, 123, 1), (2, 64, 30, 31, 62, 1)]


@pytest.mark.parametrize("shape", TEAM)
def test_channel_in_a_team(shape):
    """Also with the same bits when no member waits and each works out the sums of all others."""
    p = _Problem(*shape)
    want = p.run("local_strided")
    _same(p.run("team", 2048), want)
    if p.x.numel() < 4_000_000:  # every member reads its whole channel
        _same(p.run("team", 0), want)
    _same(p.run("team", 2048), want)
    _same(p.run("once"), want)


# more than 64 groups a channel: several waves look after their sums, in steps of four and of two
@pytest.mark.parametrize("shape", [(1, 1, 1, 640, 512, 0), (1, 2, 50, 62, 64, 1), (1, 1, 1, 460, 400, 0)])
def test_groups_that_several_waves_look_after(shape):
    """The same bits when all, some or none of the others' sums are worked out."""
    p = _Problem(*shape)
    counter = p.state.view(p.torch.int64)[:1]
    want = p.run("local_strided")
    for polls in (2048, 0, 1, 2, 3, 2048):
        _same(p.run("team", polls), want)
    assert int(counter) > 6 * 2 * 16


def test_one_state_for_doubles_and_calls_of_other_sizes():
    problems = [_Problem(*s) for s in [(2, 3, 40, 32, 32), (1, 3, 1, 64, 300), (3, 3, 17, 18, 19, 2)]]
    wants = [p.run("local_strided") for p in problems]
    for i in (0, 1, 2, 1, 0, 2):
        problems[i].state = problems[0].state
        _same(problems[i].run("team", 2048), wants[i])


def test_infinities_and_nan():
    p = _Problem(2, 4, 40, 32, 32)
    p.x[1, 1, 30, 2, 3], p.x[0, 2, 3, 4, 5], p.dy[1, 3, 7, 7, 7] = float("nan"), float("inf"), float("-inf")
    want = p.run("local_strided")
    _same(p.run("team", 2048), want)
    _same(p.run("once"), want)


@pytest.mark.parametrize("case,team", [((8, 32, 33, 33, 33, 0), True), ((32, 512, 1, 18, 18, 0), False)])
def test_a_state_is_used_where_it_is_needed(case, team):
    p = _Problem(*case)
    p.run("once")
    assert bool(p.state.any()) == team
    assert capi.load().h2x_bn_ordered_state_needed(case[0], ctypes.byref(p.geometry)) == (p.state.numel() if team else 0)


# units that do not go evenly into the groups of a channel: one more than there are, one more than twice as many; of two
# batches; teams, and workgroups that hold a channel; rows
@pytest.mark.parametrize("shape", [(9, 600, 1, 40, 30, 0), (17, 600, 1, 40, 30, 0), (70, 60, 1, 38, 38, 0), (6, 700, 1, 62, 70, 0),
                                   (35, 520, 1, 24, 23, 1), (260, 64, 1, 17, 20, 1)])
def test_units_that_do_not_go_into_the_groups(shape):
    p = _Problem(*shape)
    _same(p.run("once"), p.run("local_strided"))
