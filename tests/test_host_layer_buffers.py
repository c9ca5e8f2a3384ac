"""What the Python layers hand to the library.  Buffers that a layer makes for its launches belong to the stream it
launches on: cleared there before the launch, and on loan from that stream's memory.  On the CPU, with the
library's calls stubbed out: nothing is launched and no address is followed."""
import contextlib

import pytest

from dihydrogen_amd import capi, layers
from dihydrogen_amd.layers import BatchNormalization, HaloExchangeVirtual, Softmax, SoftmaxMode, TensorShufflerVirtual
from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor


class _Stream:
    cuda_stream = 77


class _Calls:
    """Entry points that launch nothing and say so."""

    native = capi.calls()

    def __getattr__(self, name):
        return getattr(self.native, name) if "_needed" in name else lambda *args: 0


@pytest.fixture
def made(monkeypatch):
    """(stream that was current when it was made, cleared) of every buffer."""
    current, made = [None], []

    @contextlib.contextmanager
    def on(stream):
        current.append(stream if stream is not None else current[-1])
        yield
        current.pop()

    def device_buffer(count, dtype, device="cuda", zero=False):
        import torch
        made.append((current[-1], zero))
        return torch.zeros(count, dtype=dtype)

    monkeypatch.setattr(layers.torch.cuda, "stream", on)
    monkeypatch.setattr(layers, "_device_buffer", device_buffer)
    monkeypatch.setattr(capi, "calls", _Calls)
    monkeypatch.setattr(TensorShufflerVirtual, "_plan", lambda *args: None)  # plans are made on a device
    return made


def _tensors(shape, dist, count):
    return [Tensor(shape, LocaleVirtual(r % dist.num_ranks, dist.num_ranks), dist, device="cpu").allocate()
            for r in range(count)]


def _batch_norm(stream):
    x, y, dy, dx = _tensors([40, 40, 32, 32, 2], Distribution.make_localized_distribution(5), 4)
    bn = BatchNormalization(5, 0.9, 1e-5, stream=stream)
    bn.forward(x, *[x.data] * 6, y)
    bn.backward(x, dy, *[x.data] * 7, dx)


def _softmax(stream):
    x, y, dx = _tensors([8, 4, 5, 3], Distribution.make_localized_distribution(4), 3)
    for allreduce in (None, lambda values, is_max: None):
        sm = Softmax(stream, allreduce)
        sm.setup(x, SoftmaxMode.INSTANCE)
        sm.forward(x, y)
        sm.backward(y, y, dx)


def _halo(stream):
    ranks = _tensors([8, 6, 2, 1], Distribution.make_overlapped_distribution([2, 1, 1, 1], [1, 0, 0, 0]), 2)
    xch = HaloExchangeVirtual(ranks, stream=stream)
    xch.exchange()
    xch.recv_buffer(0, 0, capi.RHS)


def _shuffle(stream):
    src, dst = _tensors([8, 6, 2, 2], Distribution([1, 1, 1, 2]), 2), _tensors([8, 6, 2, 2], Distribution([2, 1, 1, 1]), 2)
    TensorShufflerVirtual(src, dst, stream).shuffle_forward()


def _reduce(stream):
    dist = Distribution.make_localized_distribution(4)
    layers._reduce_workspaces.clear()
    layers.reduce_sum(_tensors([8, 6, 2, 2], dist, 1)[0], _tensors([1, 1, 2, 1], dist, 1)[0], stream=stream)
    layers._reduce_workspaces.clear()


@pytest.mark.parametrize("use", [_batch_norm, _softmax, _halo, _shuffle, _reduce])
def test_buffers_are_made_on_the_stream_that_is_launched_on(use, made):
    stream = _Stream()
    use(stream)
    assert made and all(s is stream for s, _ in made)
    assert any(zero for _, zero in made) == (use in (_batch_norm, _halo, _shuffle))
    made.clear()
    use(None)
    assert made and all(s is None for s, _ in made)


def test_dense_tensors_of_other_extents_go_to_the_calls_that_take_them(made, monkeypatch):
    called = []

    class Recording:
        def __getattr__(self, name):
            return lambda *args: called.append(name) or 0

    monkeypatch.setattr(capi, "calls", Recording)
    dist = Distribution.make_localized_distribution
    x = Tensor([8, 4, 6, 3], LocaleVirtual(0, 1), dist(4), device="cpu").allocate()
    for shape, forward, backward in (([4, 8, 6, 3], "local", "local"), ([8, 4, 1, 6, 3], "local", "local"),
                                     ([8, 4, 6, 3], "once", "once"), ([4, 8, 6, 2], "once", "once")):
        y = Tensor(shape, LocaleVirtual(0, 1), dist(len(shape)), device="cpu").allocate()
        bn = BatchNormalization(4, 0.9, 1e-5)
        bn.forward(x, *[x.data] * 6, y)
        bn.backward(x, y, *[x.data] * 7, x)
        assert called == ["h2x_bn_forward_" + forward, "h2x_bn_backward_" + backward]
        called.clear()


def test_what_is_packed_on_a_stream_of_its_own_is_waited_for(made, monkeypatch):
    """recv_buffer() after an exchange straight from tensor to tensor: its caller's stream waits for the packing."""
    import torch
    waited = []

    class Current:
        def wait_stream(self, stream):
            waited.append(stream)

    monkeypatch.setattr(layers.torch.cuda, "current_stream", Current)
    monkeypatch.setattr(layers, "_share_a_gpu", lambda tensors: True)

    class OnGpu(torch.Tensor):
        is_cuda = True

    monkeypatch.setattr(layers, "_device_buffer", lambda count, dtype, *args, **kwargs: torch.zeros(count, dtype=dtype).as_subclass(OnGpu))
    ranks = _tensors([8, 6, 2, 1], Distribution.make_overlapped_distribution([2, 1, 1, 1], [1, 0, 0, 0]), 2)
    stream = _Stream()
    xch = HaloExchangeVirtual(ranks, stream=stream)
    xch.exchange()
    xch.recv_buffer(0, 0, capi.RHS)
    assert waited == [stream]
    xch.recv_buffer(1, 0, capi.LHS)     # packed with the first
    assert waited == [stream]


def _normalized(layer_stream=None):
    """A batch-norm whose channels teams share, and a step of it."""
    x, y = _tensors([56, 56, 128, 16], Distribution.make_localized_distribution(4), 2)
    bn = BatchNormalization(4, 0.9, 1e-5, stream=layer_stream)

    def step():
        bn.forward(x, *[x.data] * 6, y)
        bn.backward(x, y, *[x.data] * 7, y)
    return bn, step


def _classified(layer_stream=None):
    x, y = _tensors([100, 100, 21, 2], Distribution.make_localized_distribution(4), 2)
    sm = Softmax(layer_stream)
    sm.setup(x, SoftmaxMode.INSTANCE)

    def step():
        sm.forward(x, y)
        sm.backward(y, y, x)
    return sm, step


@pytest.mark.parametrize("use", [_normalized, _classified])
def test_streams_share_no_buffer(use, made, monkeypatch):
    """Calls on two streams may run at the same time: what a launch writes to belongs to its stream.  A graph is captured
    on a stream of its own and makes nothing there."""
    current, capturing, passed = [1], [False], []
    monkeypatch.setattr(layers, "_stream_handle", lambda stream: stream.cuda_stream if stream else current[0])
    monkeypatch.setattr(layers.torch.cuda, "is_current_stream_capturing", lambda: capturing[0])

    class Calls(_Calls):
        def __getattr__(self, name):
            if "_needed" in name or "workspace_bytes" in name:
                return getattr(self.native, name)
            return lambda *args: passed.append([a.data_ptr() for a in args if a is not None and hasattr(a, "data_ptr")
                                                and id(a) in buffers] + [a for a in args if a in scalars]) or 0

    buffers, scalars = {}, set()
    device_buffer = layers._device_buffer

    def recorded(*args, **kwargs):
        b = device_buffer(*args, **kwargs)
        buffers[id(b)] = b
        scalars.add(b.data_ptr())
        return b

    monkeypatch.setattr(layers, "_device_buffer", recorded)
    monkeypatch.setattr(capi, "calls", Calls)
    layer, step = use()

    def on(stream):
        current[0] = stream
        passed.clear()
        step()
        return [set(p) for p in passed]

    first, count = on(1), len(buffers)
    second = on(2)
    assert count and len(buffers) == 2 * count
    assert all(a and not a & b for a, b in zip(first, second))
    assert on(1) == first and on(2) == second and len(buffers) == 2 * count
    capturing[0] = True
    assert on(3) == second and on(1) == first and len(buffers) == 2 * count
    capturing[0] = False
    assert not any(a & b for a, b in zip(on(3), second)) and len(buffers) == 3 * count
    # of a layer with a stream of its own, whichever is current
    layer, step = use(_Stream())
    assert on(1) == on(2)


def test_scalars_of_instance_softmax(made, monkeypatch):
    """Where a layer tells the native calls to put a sample's maximum and sum: within its buffer and apart, also in a call with fewer samples; the
    buffer is asked for its address when it is made."""
    import torch
    given, buffers, asked = [], [], []

    class Buffer(torch.Tensor):
        def data_ptr(self):
            asked.append(self)
            return super().data_ptr()

    class Recording(_Calls):
        def __getattr__(self, name):
            return (lambda *args: given.append(args) or 0) if name.endswith("_once") else super().__getattr__(name)

    def device_buffer(count, dtype, device="cuda", zero=False):
        buffers.append(torch.zeros(count, dtype=dtype).as_subclass(Buffer))
        return buffers[-1]

    monkeypatch.setattr(layers, "_device_buffer", device_buffer)
    monkeypatch.setattr(capi, "calls", Recording)
    sm = Softmax()
    dist = Distribution.make_localized_distribution(4)
    for dtype, n in ((torch.float32, 4), (torch.float32, 4), (torch.float32, 3), (torch.float32, 7), (torch.float64, 7), (torch.float64, 2)):
        x, y = (Tensor([1, 1, 10, n], LocaleVirtual(0, 1), dist, dtype, device="cpu").allocate() for _ in range(2))
        sm.setup(x, SoftmaxMode.INSTANCE)
        for backward in (False, True):
            given.clear()
            sm.backward(y, y, x) if backward else sm.forward(x, y)
            (args,), scalars = given, buffers[-1]
            first = torch.Tensor.data_ptr(scalars)
            places = [a - first for a in args if type(a) is int and 0 <= a - first < scalars.nbytes]
            assert scalars.dtype is dtype and len(places) == 2 - backward
            assert all(0 <= at <= scalars.nbytes - n * dtype.itemsize for at in places)
            assert backward or abs(places[1] - places[0]) >= n * dtype.itemsize
    assert len(asked) == 3 == len([b for b in buffers if b.dtype is not torch.uint8])
