"""What the native calls take for a pointer, and how they compare the buffers of tensors."""
import ctypes

import pytest
import torch

from dihydrogen_amd import capi
from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor


class Derived(Tensor):
    """Its interior begins elsewhere: a call asks it, not its base class."""

    def get_base_ptr(self):
        return super().get_base_ptr() + 4


def _tensor(overlap, kind=Tensor, device="cpu"):
    dist = Distribution.make_overlapped_distribution([1, 1, 1, 1], overlap)
    return kind([5, 4, 3, 2], LocaleVirtual(0, 1), dist, device=device).allocate()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [Tensor, Derived])
@pytest.mark.parametrize("overlap", [[0, 0, 0, 0], [2, 1, 0, 0]])
def test_a_local_tensor_is_the_address_of_its_interior(kind, overlap):
    t = _tensor(overlap, kind, "cuda")
    t.data.copy_(torch.arange(t.data.numel()))
    # 24 elements from there on lie in the buffer
    got, want = torch.zeros(24, device="cuda"), torch.zeros(24, device="cuda")
    for src, dst in ((t, got), (t.get_base_ptr(), want)):
        assert capi.calls().h2x_softmax_channel_forward(t.h2x_dtype, 2, 3, 4, src, dst.data_ptr(), None) == 0
    first = t.base_offset() + (kind is Derived)
    x = t.data[first:first + 24].cpu().double().view(2, 3, 4)
    assert torch.equal(got, want)
    torch.testing.assert_close(got.cpu().double().view(2, 3, 4), torch.softmax(x, 1), rtol=1e-5, atol=1e-7)


class WithBuffer(Tensor):
    """Names its allocation as torch names a tensor's; its interior is elsewhere."""

    def data_ptr(self):
        return self.get_buffer()


class Alike:
    """No Tensor, with both methods."""

    def __init__(self, t):
        self.get_base_ptr, self.data_ptr = t.get_base_ptr, t.get_buffer


@pytest.mark.parametrize("kind", ["tensor", "derived", "with data_ptr", "alike", "replaced on the object",
                                  "replaced on the class", "offset replaced on the class", "data replaced on the class"])
def test_the_address_is_what_get_base_ptr_returns(kind, monkeypatch):
    """Shown on the host: a call that reads a geometry, and geometries in the tensor's buffer."""
    # of 64 and, where the interior begins, of 128 channels, one element further on of 256
    dist = Distribution.make_overlapped_distribution([1] * 4, [1, 0, 0, 0])
    item = ctypes.sizeof(capi.TensorGeometry)
    cls = {"derived": Derived, "with data_ptr": WithBuffer}.get(kind, Tensor)
    t = cls([4096, 1, 1, 1], LocaleVirtual(0, 1), dist, torch.uint8, "cpu")
    monkeypatch.setattr(t, "base_bytes", item)
    t.allocate()
    for i, channels in enumerate((64, 128, 256)):
        g = capi.TensorGeometry()
        g.num_dims = 4
        for d, (extent, stride) in enumerate(zip((64, 64, channels, 16), (1, 64, 4096, 4096 * channels))):
            g.local_shape[d], g.strides[d] = extent, stride
        at = i * item
        t.data[at:at + item] = torch.frombuffer(bytearray(bytes(g)), dtype=torch.uint8)
    needed = capi.calls().h2x_bn_team_state_needed
    sizes = [needed(capi.F32, 16, t.get_buffer() + i * item) for i in range(3)]
    assert 0 < sizes[0] < sizes[1] < sizes[2]
    o, want = t, 1
    if kind != "derived":
        assert [needed(capi.F32, 16, t) for _ in range(2)] == [sizes[1]] * 2  # from here on the class is known as it is
    if kind == "derived":
        monkeypatch.setattr(Derived, "get_base_ptr", lambda self: Tensor.get_base_ptr(self) + item)
        want = 2
    elif kind == "alike":
        o = Alike(t)
    elif kind == "replaced on the object":
        monkeypatch.setattr(t, "get_base_ptr", lambda: t.get_buffer() + 2 * item)
        want = 2
    elif kind == "replaced on the class":
        monkeypatch.setattr(Tensor, "get_base_ptr", lambda self: self.get_buffer() + 2 * item)
        want = 2
    elif kind == "offset replaced on the class":
        monkeypatch.setattr(Tensor, "base_bytes", property(lambda self: 2 * item))
        want = 2
    elif kind == "data replaced on the class":
        later = t.data[item:]
        monkeypatch.setattr(Tensor, "data", property(lambda self: later), raising=False)
        want = 2
    assert needed(capi.F32, 16, o) == sizes[want]
    monkeypatch.undo()
    assert t.data is not None


def test_what_has_no_address_is_refused():
    t = _tensor([0, 0, 0, 0])
    t.data = None
    for p in (t, object(), "0"):
        with pytest.raises(AttributeError):
            capi.calls().h2x_softmax_channel_forward(0, 0, 0, 0, p, None, None)


def test_buffers_are_compared_in_order_and_number():
    same, ts = capi.calls().same_buffers, [_tensor([0, 0, 0, 0], kind) for kind in (Tensor, Derived, Tensor)]
    at = tuple(t.get_buffer() for t in ts)
    assert same(at, ts) and same(at, ts[:1], ts[1:]) and same((), []) and same(())
    assert not same(at, ts[:2]) and not same(at[:2], ts) and not same(at, ts[::-1]) and not same(at, ts, ts)
    ts[1].data = None
    assert not same(at, ts) and same((at[0], 0, at[2]), ts)
    ts[1].allocate()
    assert same((at[0], ts[1].get_buffer(), at[2]), ts)
    for bad in ((list(at), ts), (at, tuple(ts)), (("a", "b", "c"), ts)):
        with pytest.raises(TypeError):
            same(*bad)
    with pytest.raises(AttributeError):
        same((1,), [object()])
