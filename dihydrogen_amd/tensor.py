"""Host-side tensor model for the Python binding: distributions, virtual
locales and distributed tensors whose local parts live in torch device memory.

Mirrors the part of DistConv's tensor model the hot path is written against
(legacy/include/distconv/tensor/distribution.hpp, tensor.hpp, tensor_mpi.hpp)
with one change: the locale is *virtual* -- a (rank, size) pair without a
communicator -- so several ranks' local tensors can live on one GPU.  Shapes
and indices are innermost first, as in the reference; torch views use the
reversed (outermost first) order.
"""
from __future__ import annotations

import ctypes
import math
from typing import Iterable, List, Optional, Sequence

import torch

from . import capi


def _prod(values: Iterable[int]) -> int:
    return math.prod(int(v) for v in values)


class Distribution:
    """legacy/include/distconv/tensor/distribution.hpp:14-275."""

    def __init__(self, locale_shape: Sequence[int], split_shape: Optional[Sequence[int]] = None,
                 overlap: Optional[Sequence[int]] = None):
        self.locale_shape = [int(v) for v in locale_shape]
        self.split_shape = list(self.locale_shape) if split_shape is None else [int(v) for v in split_shape]
        nd = len(self.locale_shape)
        ov = [0] * nd if overlap is None else [int(v) for v in overlap]
        if len(self.split_shape) != nd or len(ov) != nd:
            raise ValueError("locale shape, split shape and overlap must have the same length")
        for l, s in zip(self.locale_shape, self.split_shape):
            if s < 1 or l % s != 0:
                raise ValueError(f"locale extent {l} is not divisible by split extent {s}")
        # halo only where the dimension is actually split (distribution.hpp:245-251)
        self.overlap = [o if s > 1 else 0 for o, s in zip(ov, self.split_shape)]

    # factories, named as in the reference (distribution.hpp:54-95)
    @staticmethod
    def make_localized_distribution(num_dims: int) -> "Distribution":
        return Distribution([1] * num_dims)

    @staticmethod
    def make_distribution(locale_shape: Sequence[int]) -> "Distribution":
        return Distribution(locale_shape)

    @staticmethod
    def make_overlapped_distribution(locale_shape, overlap) -> "Distribution":
        return Distribution(locale_shape, locale_shape, overlap)

    @staticmethod
    def make_shared_distribution(locale_shape, split_shape=None) -> "Distribution":
        return Distribution(locale_shape, [1] * len(locale_shape) if split_shape is None else split_shape)

    @property
    def num_dims(self) -> int:
        return len(self.locale_shape)

    @property
    def num_ranks(self) -> int:
        return _prod(self.locale_shape)

    def get_num_ranks_per_split(self, dim: int) -> int:
        return self.locale_shape[dim] // self.split_shape[dim]

    def is_distributed(self, dim: int) -> bool:
        return self.split_shape[dim] > 1

    def is_split_root_index(self, rank_index: Sequence[int]) -> bool:
        return all(r % self.get_num_ranks_per_split(d) == 0 for d, r in enumerate(rank_index))

    def rank_index(self, rank: int) -> List[int]:
        """rank -> grid index, dimension 0 fastest (tensor_mpi.hpp:47-56)."""
        out = []
        for extent in self.locale_shape:
            rank, r = divmod(rank, extent)
            out.append(r)
        return out

    def rank_of(self, rank_index: Sequence[int]) -> int:
        rank = 0
        for extent, r in zip(reversed(self.locale_shape), reversed(list(rank_index))):
            rank = rank * extent + r
        return rank

    def __eq__(self, other):
        return (isinstance(other, Distribution) and self.locale_shape == other.locale_shape
                and self.split_shape == other.split_shape and self.overlap == other.overlap)


class LocaleVirtual:
    """Stands in for LocaleMPI (tensor_mpi.hpp:16-90): a rank among `size`
    ranks that all live in this process."""

    def __init__(self, rank: int, size: int):
        if not 0 <= rank < size:
            raise ValueError("rank out of range")
        self.rank, self.size = rank, size

    def get_rank(self) -> int:
        return self.rank

    def get_size(self) -> int:
        return self.size


def _block_start(extent: int, parts: int, index: int) -> int:
    """First element of part `index` when `extent` is cut into `parts` blocks,
    the first extent % parts of which are one longer (tensor_mpi.hpp:458-488)."""
    base, rem = divmod(extent, parts)
    return index * base + min(index, rem)


_TORCH_DTYPES = {torch.float32: capi.F32, torch.float64: capi.F64}


class _once:
    """A property that is worked out at its first use and then an attribute of the instance
    (functools.cached_property takes a lock to do so)."""

    def __init__(self, compute):
        self.compute, self.name = compute, compute.__name__
        self.__doc__ = compute.__doc__

    def __get__(self, instance, owner=None):
        if instance is None:
            return self
        value = instance.__dict__[self.name] = self.compute(instance)
        return value


class Layout:
    """What a layer call needs to know about a local tensor besides its address.  Shape,
    distribution and type of a Tensor are fixed when it is made, so this is worked out once
    (a layer call that launches a kernel of a few microseconds cannot afford it every time), and
    what only some calls need when one of them does: a tensor may be new at every call."""

    def __init__(self, t: "Tensor"):
        local, real, overlap, shape, dist = t.local_shape, t.local_real_shape, t.overlap, t.shape, t.dist
        self._local, self._real, self._overlap = local, real, overlap
        ns = len(local) - 2
        spatial = spatial_real = 1
        for d in range(ns):
            spatial *= local[d]
            spatial_real *= real[d]
        self.spatial, self.spatial_real = spatial, spatial_real
        samples, channels = self.samples, self.channels = local[ns + 1], local[ns]
        self.extents = tuple(local[:ns + 1])  # of one sample
        # no halo on the inner spatial dimensions: the layout the dense entry points take
        # (legacy/src/dnn_backend/batchnorm.cu:210-219)
        self.dense = not any(overlap[:max(ns - 1, 0)])
        self.haloed = any(overlap)
        self.channel_halo = overlap[ns] != 0 or overlap[ns + 1] != 0
        self.dtype = _TORCH_DTYPES[t.dtype]
        # a rank that owns elements
        self.active = spatial * samples * channels > 0 and (dist.locale_shape == dist.split_shape or t.is_split_root())
        # elements per channel of the local and of the global shape
        self.per_channel_local = spatial * samples if channels else 0
        self.per_channel_global = math.prod(shape) // shape[ns] if shape[ns] else 0
        # channels that no workgroups share: up to 16 K floats or 4 K doubles
        self.small_channels = samples * spatial_real <= (4096 if self.dtype == capi.F64 else 16384)

    @_once
    def alike(self):
        """Tensors with equal keys lie in memory alike."""
        return tuple(self._local), tuple(self._real), tuple(self._overlap), self.dtype

    @_once
    def geometry(self):
        """h2x_tensor_geometry: local extents and the strides of the real allocation."""
        g = capi.TensorGeometry()
        nd = g.num_dims = len(self._local)
        strides, stride = [], 1
        for extent in self._real:
            strides.append(stride)
            stride *= extent
        g.local_shape[:nd] = self._local
        g.strides[:nd] = strides
        return g

    @_once
    def geometry_address(self) -> int:
        return ctypes.addressof(self.geometry)

    @_once
    def team_state_bytes(self) -> int:
        """State for batch-norm calls on tensors like this (0: none is for teams of workgroups)."""
        return capi.calls().h2x_bn_team_state_needed(self.dtype, self.samples, self.geometry_address)

    @_once
    def ordered_state_bytes(self) -> int:
        """The same for calls on double tensors, whose teams add in the order of the staged calls."""
        return capi.calls().h2x_bn_ordered_state_needed(self.samples, self.geometry_address)

    @_once
    def instance_state_bytes(self) -> int:
        """State for instance softmax of tensors like this (0: no workgroups share a sample)."""
        return capi.calls().h2x_softmax_instance_state_needed(self.dtype, self.samples, self.channels * self.spatial)

    @_once
    def instance_workspace_bytes(self) -> int:
        return capi.calls().h2x_softmax_instance_workspace_bytes(self.samples)

    @_once
    def clearing_team_state_bytes(self) -> int:
        """The same for calls that clear their output's halo."""
        return capi.calls().h2x_bn_team_state_needed_clearing(self.dtype, self.haloed_geometry_address)

    @_once
    def haloed_geometry(self):
        """h2x_haloed_geometry: local and real extents, halo widths."""
        g = capi.HaloedGeometry()
        nd = g.num_dims = len(self._local)
        g.local_shape[:nd], g.real_shape[:nd], g.lower_halo[:nd] = self._local, self._real, self._overlap
        return g

    @_once
    def haloed_geometry_address(self) -> int:
        return ctypes.addressof(self.haloed_geometry)


class Tensor:
    """Tensor<DataType, LocaleVirtual, device allocator>: global shape plus
    distribution; `allocate()` creates the local real (haloed) buffer."""

    def __init__(self, shape: Sequence[int], locale: LocaleVirtual, dist: Distribution,
                 dtype: torch.dtype = torch.float32, device: str = "cuda"):
        self.shape = [int(v) for v in shape]
        if len(self.shape) != dist.num_dims:
            raise ValueError("shape and distribution disagree on the number of dimensions")
        if math.prod(dist.locale_shape) != locale.size:
            raise ValueError("distribution does not cover the locale")
        self.locale, self.dist, self.dtype, self.device = locale, dist, dtype, device
        self.proc_index = dist.rank_index(locale.rank)
        self.split_index = [p // (l // s) for p, l, s in zip(self.proc_index, dist.locale_shape, dist.split_shape)]
        self.global_index, self.local_shape = [], []
        for extent, parts, index in zip(self.shape, dist.split_shape, self.split_index):
            lo, hi = 0, extent
            if parts > 1:
                lo, hi = _block_start(extent, parts, index), _block_start(extent, parts, index + 1)
            self.global_index.append(lo)
            self.local_shape.append(hi - lo)
        self.overlap = list(dist.overlap)
        self.local_real_shape = [l + 2 * o for l, o in zip(self.local_shape, self.overlap)]
        self.data: Optional[torch.Tensor] = None

    # -- geometry ------------------------------------------------------------
    def get_num_dims(self) -> int:
        return len(self.shape)

    def get_local_size(self) -> int:
        return _prod(self.local_shape)

    def get_local_real_size(self) -> int:
        return _prod(self.local_real_shape)

    def is_split_root(self) -> bool:
        return self.dist.is_split_root_index(self.proc_index)

    def get_strides(self) -> List[int]:
        """tensor.hpp:291-298."""
        out, s = [], 1
        for extent in self.local_real_shape:
            out.append(s)
            s *= extent
        return out

    def get_dimension_rank_offset(self, dim: int, rank_index: int) -> int:
        parts = self.dist.split_shape[dim]
        if parts == 1:
            return 0
        return _block_start(self.shape[dim], parts, rank_index // self.dist.get_num_ranks_per_split(dim))

    def get_remote_dimension(self, dim: int, rank_index: int) -> int:
        parts = self.dist.split_shape[dim]
        if parts == 1:
            return self.shape[dim]
        si = rank_index // self.dist.get_num_ranks_per_split(dim)
        return _block_start(self.shape[dim], parts, si + 1) - _block_start(self.shape[dim], parts, si)

    @_once
    def layout(self) -> Layout:
        return Layout(self)

    @_once
    def base_bytes(self) -> int:
        return self.base_offset() * self.dtype.itemsize

    def base_offset(self) -> int:
        return sum(o * s for o, s in zip(self.overlap, self.get_strides()))

    @property
    def h2x_dtype(self) -> int:
        return _TORCH_DTYPES[self.dtype]

    # -- storage -------------------------------------------------------------
    def allocate(self) -> "Tensor":
        self.data = torch.zeros(max(self.get_local_real_size(), 1), dtype=self.dtype, device=self.device)
        return self

    def get_buffer(self) -> int:
        """Device address of the real allocation (tensor.hpp:449-460)."""
        return self.data.data_ptr()

    def get_base_ptr(self) -> int:
        """Device address of the first interior element (tensor.hpp:462-481)."""
        return self.data.data_ptr() + self.base_bytes

    def real_view(self) -> torch.Tensor:
        """The real local tensor as a torch view, outermost dimension first."""
        n = self.get_local_real_size()
        return self.data[:n].view(*reversed(self.local_real_shape))

    def interior_view(self) -> torch.Tensor:
        v = self.real_view()
        for axis, (o, l) in enumerate(zip(reversed(self.overlap), reversed(self.local_shape))):
            v = v.narrow(axis, o, l)
        return v


# what the native module does by itself for a tensor that has no others (csrc/h2x_python.cpp)
BASE_PTR_PARTS = Tensor.get_base_ptr, Tensor.base_bytes
