"""The state through which workgroups that share a channel exchange its sums is asked for, and made by the layers,
where a call uses it and not otherwise."""
import ctypes

import pytest

from dihydrogen_amd import capi
from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor

# N, C, D, H, W, halo; a state is needed
CASES = [((8, 64, 1, 56, 56, 0), True), ((4, 64, 64, 64, 64, 0), True), ((8, 64, 30, 30, 30, 1), True),
         ((32, 512, 1, 28, 28, 0), False),          # one workgroup holds a channel, and channels are many
         ((2048, 256, 1, 7, 7, 0), False),          # short segments
         ((2, 2, 40, 20, 20, 0), False),            # too few workgroups
         ((100, 64, 64, 64, 64, 0), False),         # more than a team holds
         ((64, 4096, 1, 30, 30, 0), False)]


def _tensor(n, c, d, h, w, halo, dtype=None):
    import torch
    split = 2 if halo else 1
    spatial = [w, h] + ([d] if d > 1 else [])
    dist = Distribution.make_overlapped_distribution([split] * len(spatial) + [1, 1], [halo] * len(spatial) + [0, 0])
    return Tensor([e * split for e in spatial] + [c, n], LocaleVirtual(0, dist.num_ranks), dist,
                  dtype or torch.float32, device="cpu")


@pytest.mark.parametrize("case,needed", CASES)
def test_state_needed(case, needed):
    import torch
    lib, c = capi.load(), case[1]
    layout = _tensor(*case).layout
    assert layout.team_state_bytes == (lib.h2x_bn_team_state_bytes(c) if needed else 0)
    if case[5]:
        assert layout.clearing_team_state_bytes == (lib.h2x_bn_team_state_bytes(c) if needed else 0)
    double = _tensor(*case, torch.float64).layout
    assert double.team_state_bytes == double.clearing_team_state_bytes == 0
    assert lib.h2x_bn_team_state_needed(capi.F32, 1, None) == lib.h2x_bn_team_state_needed_clearing(capi.F32, None) == 0
    bad = capi.TensorGeometry.from_buffer_copy(layout.geometry)
    bad.num_dims = 7
    assert lib.h2x_bn_team_state_needed(capi.F32, case[0], ctypes.byref(bad)) == 0


@pytest.mark.parametrize("case,needed", CASES[:3] + CASES[3:4] + CASES[5:6])
def test_layers_make_a_state_where_it_is_used(case, needed, monkeypatch):
    import torch
    from dihydrogen_amd import layers

    native = capi.calls()

    class Calls:
        def __getattr__(self, name):
            return getattr(native, name) if "_needed" in name else lambda *args: 0

    monkeypatch.setattr(capi, "calls", Calls)
    monkeypatch.setattr(layers, "_device_buffer", lambda count, dtype, device="cuda", zero=False: torch.zeros(count, dtype=dtype))
    x = _tensor(*case)
    x.data = torch.zeros(1)                         # no address is followed
    for clear in (False, True):
        bn = layers.BatchNormalization(x.get_num_dims(), 0.9, 1e-5, clear_output_halo=clear)
        bn.forward(x, *[x.data] * 6, x)
        bn.backward(x, x, *[x.data] * 7, x)
        assert (bn._state is not None) == needed


def test_size_of_a_state():
    """Room for 256 sums a channel, 512 for the first 32: of more channels no call has larger teams."""
    lib = capi.load()
    size = lib.h2x_bn_team_state_bytes
    assert size(2048) <= 2048 * (128 + 256 * 16) + 32 * 256 * 16 + 256
    assert [size(c + 1) - size(c) for c in (1, 31, 32, 2047)] == [8320, 8320, 4224, 4224]
    # 71 members of 128 KB a channel backward: such channels are more than 8 MB, and a tensor of them that takes teams has few
    assert _tensor(17, 27, 1, 368, 368, 0).layout.team_state_bytes == size(27)
