"""Softmax of samples that a wave or a workgroup holds, by their number: at the edges of the rule that chooses between the two, against float64."""
import pytest

import test_gpu_softmax_rows as rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("kind", ["instance", "channel"])
@pytest.mark.parametrize("n", [512, 768, 769, 2048, 2049])
def test_numbers_of_samples(n, kind, dtype):
    for size in (256, 257, 512, 513, 1025, 2048):
        rows._check(kind, n, size, dtype)


@pytest.mark.parametrize("size", [257, 300, 400, 512])
def test_rows_by_waves(size):
    """Channel softmax of floats, forward, 257 to 512 channels: from 513 samples on a sample's bits are those that a wave gives it in a large batch."""
    import torch
    from dihydrogen_amd import capi
    calls, st = capi.calls(), torch.cuda.current_stream().cuda_stream
    x = torch.randn((1500, size), device="cuda", generator=torch.Generator(device="cuda").manual_seed(size)) * 2
    many, few = torch.empty_like(x), torch.empty_like(x)
    assert calls.h2x_softmax_channel_forward(capi.F32, 1500, size, 1, x, many, st) == 0
    for n in (513, 700, 768, 769):
        assert calls.h2x_softmax_channel_forward(capi.F32, n, size, 1, x, few, st) == 0
        assert torch.equal(few[:n], many[:n]), n
