"""Batch-norm between dense tensors whose local extents differ but pair up in order (H x W and W x H, 4-D and 5-D
with one plane, a larger batch's buffer): done as by the staged calls, bit for bit."""
import pytest

pytestmark = pytest.mark.gpu

# innermost first: input, output (d_output, d_input)
SHAPES = [([8, 4, 6, 3], [4, 8, 6, 3]), ([8, 4, 1, 6, 3], [8, 4, 6, 3]), ([8, 4, 6, 3], [32, 1, 1, 6, 3]),
          ([90, 70, 5, 2], [70, 90, 5, 4]), ([8, 4, 6, 3], [8, 5, 6, 3])]


def _run(shapes, dtype, fuse_local):
    import torch
    from dihydrogen_amd.layers import BatchNormalization
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    g = torch.Generator(device="cuda").manual_seed(4)
    x, y, dy, dx = (Tensor(s, LocaleVirtual(0, 1), Distribution.make_localized_distribution(len(s)), dtype).allocate()
                    for s in (shapes[0], shapes[1], shapes[1], shapes[1]))
    for t in (x, dy):
        t.data.normal_(0.5, 1, generator=g)
    c = shapes[0][-2]
    v = [torch.full((c,), float(i), dtype=dtype, device="cuda") for i in range(1, 11)]
    bn = BatchNormalization(len(shapes[0]), 0.9, 1e-5, fuse_local=fuse_local)
    bn.forward(x, *v[:6], y)
    bn.backward(x, dy, v[0], v[1], v[4], *v[6:], dx)
    torch.cuda.synchronize()
    return [y.data, dx.data] + v


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("shapes", SHAPES)
def test_as_the_staged_calls(shapes, dtype):
    import torch
    for a, b in zip(_run(shapes, getattr(torch, dtype), True), _run(shapes, getattr(torch, dtype), False)):
        assert torch.equal(a, b)


def test_extents_that_would_leave_the_memory_are_refused():
    import torch
    from dihydrogen_amd.capi import H2XError
    with pytest.raises(H2XError):
        _run(([8, 4, 6, 3], [4, 8, 6, 2]), torch.float32, True)
