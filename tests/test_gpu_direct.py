"""Tensor-to-tensor launches (halo exchange of a whole grid, reverse exchange, clearing, shuffle) against the
packed path - receive buffers, arenas - bit for bit, from tensors filled with different values everywhere,
halos included."""
import numpy as np
import pytest

import test_host_direct_launch_audit as audits

pytestmark = pytest.mark.gpu


def _tensors(shape, locale, split, overlap, dtype, seed):
    import torch
    from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor
    n = int(np.prod(locale))
    g = torch.Generator(device="cuda").manual_seed(seed)
    ts = [Tensor(shape, LocaleVirtual(r, n), Distribution(locale, split, overlap), dtype).allocate() for r in range(n)]
    for t in ts:
        if dtype.is_floating_point:
            t.data.uniform_(-1, 1, generator=g)
        else:
            t.data.random_(-30000, 30000, generator=g)
    return ts


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("case", audits.GRIDS)
def test_grid_launches_equal_the_packed_exchange(case, periodic, dtype):
    import torch
    from dihydrogen_amd.layers import HaloExchangeAccumOp, HaloExchangeVirtual
    shape, locale, overlap = case
    steps = {op.name: (lambda x, op=op: x.exchange(is_reverse=True, op=op)) for op in HaloExchangeAccumOp}
    steps["forward"] = lambda x: x.exchange()
    steps["clear"] = lambda x: x.clear_halos()
    steps["conv input"] = lambda x: (x.clear_halos(only_unfilled=True), x.exchange())
    for name, step in steps.items():
        a, b = (_tensors(shape, locale, None, overlap, getattr(torch, dtype), 5) for _ in range(2))
        xa, xb = HaloExchangeVirtual(a, periodic=periodic), HaloExchangeVirtual(b, periodic=periodic)
        assert xa._grid(1)
        if name in HaloExchangeAccumOp.__members__ and not xa._grid(2):
            continue    # boundary strips that share cells: packed on both sides
        xb._grid_of = (xb._addresses(), 0, -1)      # as where the tensors do not share a GPU
        step(xa), step(xb)
        assert not xa._recv
        torch.cuda.synchronize()
        for ta, tb in zip(a, b):
            assert torch.equal(ta.data, tb.data), name


@pytest.mark.parametrize("dtype", ["float32", "int16", "float64"])
def test_direct_shuffles_equal_the_packed_ones(dtype, monkeypatch):
    import torch
    import test_gpu_shuffle as cases
    from dihydrogen_amd import layers
    for name, (shape, (sl, ss, so), (dl, ds, do)) in cases.CASES.items():
        results = []
        for direct in (True, False):
            with monkeypatch.context() as m:
                if not direct:
                    m.setattr(layers, "_share_a_gpu", lambda tensors: False)
                src, dst = (_tensors(shape, *side, getattr(torch, dtype), seed)
                            for seed, side in ((1, (sl, ss, so)), (2, (dl, ds, do))))
                sh = layers.TensorShufflerVirtual(src, dst)
            assert (sh._direct_plan is not None) == direct, name
            sh.shuffle_forward()
            torch.cuda.synchronize()
            results.append([t.data.clone() for t in dst])
            for t in src:
                t.data.zero_()
            sh.shuffle_backward()
            torch.cuda.synchronize()
            results[-1] += [t.data for t in src]
        for ta, tb in zip(*results):
            assert torch.equal(ta, tb), name


def test_a_shuffle_whose_source_lies_in_its_destination_is_packed():
    import torch
    from dihydrogen_amd import layers
    src = _tensors((8, 8, 2, 4), (1, 1, 1, 4), None, None, torch.float32, 1)
    dst = _tensors((8, 8, 2, 4), (2, 2, 1, 1), None, None, torch.float32, 2)
    want = _tensors((8, 8, 2, 4), (2, 2, 1, 1), None, None, torch.float32, 2)
    layers.TensorShufflerVirtual(src, want).shuffle_forward()
    for s, d in zip(src, dst):
        d.data = s.data                             # in place
    sh = layers.TensorShufflerVirtual(src, dst)
    sh.shuffle_forward()
    torch.cuda.synchronize()
    for d, w in zip(dst, want):
        assert torch.equal(d.data, w.data)
