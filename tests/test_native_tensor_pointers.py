"""The address that a native call takes of a torch tensor: what its data_ptr() returns, or raises.  Shown on the host, by a call that
reads a geometry out of the tensor's memory."""
import ctypes

import pytest
import torch

from dihydrogen_amd import capi

ITEM = ctypes.sizeof(capi.TensorGeometry)


class Shifted(torch.Tensor):
    """One item further on."""

    def data_ptr(self):
        return super().data_ptr() + ITEM


def _geometries():
    """The bytes of a geometry that teams have a state for, and of one with twice the channels; the states."""
    raw, needed = bytearray(), []
    for c in (64, 128):
        g = capi.TensorGeometry()
        g.num_dims = 4
        g.local_shape[:4] = 64, 64, c, 16
        g.strides[:4] = 1, 64, 4096, 4096 * c
        raw += bytes(g)
        needed.append(capi.calls().h2x_bn_team_state_needed(capi.F32, 16, ctypes.addressof(g)))
    assert len(raw) == 2 * ITEM and 0 < needed[0] < needed[1]
    return torch.frombuffer(raw, dtype=torch.uint8), needed


def _needed(pointer):
    return capi.calls().h2x_bn_team_state_needed(capi.F32, 16, pointer)


def test_tensors_views_and_parameters():
    t, (first, second) = _geometries()
    assert _needed(t) == _needed(t.data_ptr()) == first
    assert _needed(t[ITEM:]) == second
    assert _needed(torch.nn.Parameter(t[ITEM:], requires_grad=False)) == second


def test_a_class_with_a_data_ptr_of_its_own_is_asked():
    t, (first, second) = _geometries()
    assert _needed(t.as_subclass(Shifted)) == second


def test_a_tensor_without_memory_raises_what_data_ptr_raises():
    messages = []

    def asked(x):
        for ask in (lambda: x.data_ptr(), lambda: _needed(x)):
            with pytest.raises(RuntimeError) as e:
                ask()
            messages.append(str(e.value))
        return x

    torch.func.vmap(asked)(torch.zeros(2, 3))
    assert messages[0] == messages[1]


def test_only_the_torch_that_the_module_was_compiled_for_is_read_directly():
    """Another torch may have its tensors' addresses elsewhere: they are asked by their method."""
    from dihydrogen_amd.tensor import BASE_PTR_PARTS, Tensor
    t, (first, second) = _geometries()
    told = lambda version, sample=t: capi.calls().pointer_types(torch.Tensor, Tensor, *BASE_PTR_PARTS, version, sample)
    try:
        for version in ("2.0.0", torch.__version__ + ".1", torch.__version__[:-1], ""):
            assert told(version) is False
            assert (_needed(t), _needed(t[ITEM:])) == (first, second)
        assert told(torch.__version__, t.as_subclass(Shifted)) is False
    finally:
        assert told(torch.__version__) is True
    assert (_needed(t), _needed(t[ITEM:])) == (first, second)


def test_a_mode_is_told_of_the_call():
    from torch.overrides import TorchFunctionMode
    t, (first, second) = _geometries()

    class Further(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {})) + (ITEM if func is torch.Tensor.data_ptr else 0)

    with Further():
        assert _needed(t) == second
        with torch._C.DisableTorchFunction():
            assert _needed(t) == first
    assert _needed(t) == first


def test_a_replaced_data_ptr_is_asked(monkeypatch):
    t, (first, second) = _geometries()
    own = torch.Tensor.data_ptr
    for _ in range(2):
        with monkeypatch.context() as m:
            m.setattr(torch.Tensor, "data_ptr", lambda self: own(self) + ITEM)
            assert _needed(t) == second
        assert _needed(t) == first
        with monkeypatch.context() as m:
            m.setattr(torch.Tensor, "unrelated", 1, raising=False)
            assert _needed(t) == first
    t.unrelated = 1
    assert _needed(t) == first
    t.data_ptr = lambda: own(t) + ITEM
    assert _needed(t) == second
    del t.data_ptr
    assert _needed(t) == first


def test_a_replaced_data_ptr_of_local_tensors_data_is_asked(monkeypatch):
    """Through a local tensor, whose get_base_ptr() the native module plays, and in the comparison of buffers."""
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    t, (first, second) = _geometries()
    local = Tensor([t.numel()], LocaleVirtual(0, 1), Distribution.make_localized_distribution(1), torch.uint8, device="cpu")
    local.data = t
    local.base_bytes
    own = torch.Tensor.data_ptr
    assert _needed(local) == first and capi.calls().same_buffers((own(t),), [local])
    monkeypatch.setattr(torch.Tensor, "data_ptr", lambda self: own(self) + ITEM)
    assert _needed(local) == second and capi.calls().same_buffers((own(t) + ITEM,), [local])
