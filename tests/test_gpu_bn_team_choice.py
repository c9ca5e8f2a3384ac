"""How many workgroups share a channel, by what they count in the state of its first channel: 0 where a pass runs in two launches
or by one workgroup a channel."""
import ctypes

import pytest

import test_gpu_bn_once as once
from dihydrogen_amd import capi

pytestmark = pytest.mark.gpu


def _forward_members(p):
    """Of a forward pass of the float problem p."""
    lib, torch, t = capi.load(), p.torch, lambda v: v.data_ptr()
    gp, at = ctypes.byref(p.geometry), lambda v: v.data_ptr() + p.offset
    vec = [torch.ones_like(p.scale) for _ in range(4)]
    y = torch.empty_like(p.x)
    p.state.zero_()
    status = lib.h2x_bn_forward_once(capi.F32, p.n, gp, gp, at(p.x), t(p.scale), t(p.bias), p.per, 0.9, 1e-5, *[t(v) for v in vec],
                                     at(y), t(p.ws), t(p.state), torch.cuda.current_stream().cuda_stream)
    assert status == 0
    torch.cuda.synchronize()
    return int(p.state.view(torch.int64)[0])


def _backward_members(p):
    """Of a backward pass of the float problem p."""
    lib, torch, t = capi.load(), p.torch, lambda v: v.data_ptr()
    gp, at = ctypes.byref(p.geometry), lambda v: v.data_ptr() + p.offset
    vec = [torch.ones_like(p.scale) for _ in range(6)]
    dx = torch.empty_like(p.x)
    p.state.zero_()
    status = lib.h2x_bn_backward_once(capi.F32, p.n, p.per, gp, gp, gp, at(p.x), at(p.dy), t(vec[0]), t(vec[1]), t(p.scale),
                                      *[t(v) for v in vec[2:]], at(dx), 1e-5, t(p.ws), t(p.state),
                                      torch.cuda.current_stream().cuda_stream)
    assert status == 0
    torch.cuda.synchronize()
    return int(p.state.view(torch.int64)[0])


# N, C, D, H, W, halo: 128 members of a dense channel of 16 MB; 98 with a halo, and 67 and 88 in larger tensors
@pytest.mark.parametrize("shape,members", [((16, 2, 64, 64, 64, 0), 128), ((100, 8, 1, 200, 160, 1), 98),
                                           ((158, 13, 25, 23, 21, 1), 0), ((14, 11, 65, 66, 48, 2), 0)])
def test_large_teams_backward(shape, members):
    assert _backward_members(once._Problem(*shape)) == members


# 2000 members of 64 KB would be 2.6 rounds of the chip; 64 members a channel are one; a handful is left to two launches; one
# workgroup holds the last
@pytest.mark.parametrize("shape,members", [((4, 16, 96, 63, 84, 0), 63), ((4, 64, 64, 64, 64, 0), 32), ((8, 64, 1, 56, 56, 0), 4),
                                           ((2, 2, 40, 20, 20, 0), 0), ((32, 512, 1, 28, 28, 0), 0)])
def test_forward(shape, members):
    assert _forward_members(once._Problem(*shape)) == members


# members of 64 KB of each tensor, one round of the chip, not three of 32 KB a CU; long haloed rows above 104 MiB
@pytest.mark.parametrize("shape,members", [((120, 48, 8, 10, 12, 1), 8), ((250, 90, 1, 16, 15, 1), 4), ((4, 8, 96, 96, 96, 1), 108)])
def test_backward_with_a_halo(shape, members):
    assert _backward_members(once._Problem(*shape)) == members


@pytest.mark.parametrize("shape,members", [((76, 6, 18, 21, 20, 0), 36), ((32, 256, 1, 56, 56, 0), 4)])
def test_forward_in_larger_members(shape, members):
    assert _forward_members(once._Problem(*shape)) == members
