"""What h2x_bn_team_state_needed says is what the calls do: a state is written to where it is needed, and only
there."""
import ctypes

import pytest

import test_gpu_bn_once as once
import test_host_bn_team_state as host
from dihydrogen_amd import capi

pytestmark = pytest.mark.gpu

# (channels beyond a gigabyte left out)
SHAPES = [(*s, 0) for s in once.ONCE] + once.TEAM + [c for c, _ in host.CASES if c[0] * c[1] * c[2] * c[3] * c[4] < 2 ** 28]


@pytest.mark.parametrize("shape", SHAPES)
def test_a_state_is_used_where_it_is_needed(shape):
    p = once._Problem(*shape)
    assert not p.state.any()
    p.run("once")
    needed = capi.load().h2x_bn_team_state_needed(capi.F32, shape[0], ctypes.byref(p.geometry))
    assert bool(p.state.any()) == (needed > 0)
    assert needed in (0, p.state.numel())


def test_one_state_for_the_largest_teams_and_more_channels():
    """Channels beyond the 32nd have room for half as many sums as those before them; where a channel's lie is one place for
    all calls."""
    shapes = [(17, 3, 1, 368, 368), (8, 40, 1, 56, 56), (4, 33, 1, 66, 68), (17, 3, 1, 368, 368), (8, 64, 1, 56, 56)]
    problems = [once._Problem(*s) for s in shapes]
    wants = [p.run("local_strided") for p in problems]
    for k in (0, 1, 2, 3, 4, 0, 4, 1):
        problems[k].state = problems[4].state
        once._close(problems[k].run("once"), wants[k])
