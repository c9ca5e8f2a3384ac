"""Channels that one workgroup would hold, by teams or by that workgroup: what they count in the state of the first channel, around
the sizes where the rule changes, and the results of either as the two-launch calls'."""
import pytest

import test_gpu_bn_once as once
import test_gpu_bn_team_choice as choice

pytestmark = pytest.mark.gpu

# N, C, D, H, W, halo; teams.  8192 and more vectors, channels that fill rounds of workgroups or do not, more channels than a state is for
SHAPES = [((8, 128, 1, 64, 64, 0), False), ((8, 128, 1, 64, 65, 0), True), ((16, 130, 1, 56, 56, 0), True),
          ((8, 300, 1, 56, 56, 0), True), ((8, 400, 1, 56, 56, 0), False), ((7, 530, 1, 56, 56, 0), True),
          ((3, 300, 12, 13, 15, 1), False), ((8, 300, 12, 13, 15, 1), True), ((9, 2049, 1, 61, 61, 0), False)]


@pytest.mark.parametrize("shape,teams", SHAPES)
def test_who_shares_a_channel(shape, teams):
    p = once._Problem(*shape)
    assert (choice._forward_members(p) > 0) == teams
    once._close(p.run("once"), p.run("local_strided"))
