"""Python mirror of the DistConv layer API for the non-convolution hot path,
on top of the C ABI (``include/h2x.h``).  Method names, argument order and
return values follow the reference classes; MPI ranks are replaced by virtual
ranks whose local tensors live on one GPU, and every "transfer" between ranks
is pointer wiring between device buffers.
"""
from __future__ import annotations

import ctypes
from enum import Enum
from typing import Callable, List, Optional, Sequence

import torch

from . import capi
from .tensor import Layout, Tensor, _prod


def _device_buffer(count: int, dtype, device="cuda", zero: bool = False) -> torch.Tensor:
    """Every device buffer the layers own (workspaces, receive buffers, the shuffler's arena)
    comes from here, so that a test can put guard zones around them."""
    return (torch.zeros if zero else torch.empty)(count, dtype=dtype, device=device)


def _buffer_of(stream: Optional[torch.cuda.Stream], *args, **kwargs) -> torch.Tensor:
    """A _device_buffer for launches on `stream` (None: on the current one).  It is made on that
    stream: what clears it comes before the launches that use it, and whoever gets its memory when
    the layer gives it back comes after them.  On another stream neither would be ordered."""
    if stream is None:
        return _device_buffer(*args, **kwargs)
    with torch.cuda.stream(stream):
        return _device_buffer(*args, **kwargs)


def _share_a_gpu(tensors: Sequence[Tensor]) -> bool:
    """All tensors are allocated, on one GPU: what belongs to another rank can be read and written
    where it lies.  (On the host, where launches can only be audited, strips are packed as they
    would be for a transport.)"""
    first = tensors[0].data
    return all(t.data is not None and t.data.is_cuda and t.data.device == first.device for t in tensors)


_has_gpu: Optional[bool] = None
_current_device = _current_stream = None  # torch's bindings, once there is a GPU


def _stream_handle(stream: Optional[torch.cuda.Stream]) -> int:
    """Handle of `stream`, or of the current stream of the current device (asked of torch's
    bindings directly: torch.cuda.current_stream() makes an object first, 2.8 us against 0.2)."""
    if stream is not None:
        return stream.cuda_stream
    if _current_stream is not None:
        return _current_stream(_current_device())
    return _first_stream_handle()


def _first_stream_handle() -> int:
    global _has_gpu, _current_device, _current_stream
    if _has_gpu is None:
        _has_gpu = torch.cuda.is_available()  # asked once: the answer does not change
        if _has_gpu:
            torch.cuda.init()
    if not _has_gpu:
        # no GPU: the null stream; every launch then fails with HIP's own error.  (Launch
        # audits, which play the kernels' indexing on the CPU, ignore the stream.)
        return 0
    _current_device, _current_stream = torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream
    return _current_stream(_current_device())


class _Kept:
    """What a layer keeps for its calls on one stream, each buffer behind what it is for: calls on other streams,
    which may run at the same time, have their own.  (A tuple is replaced as a whole: threads may share a layer.)"""
    __slots__ = ("workspace", "scalars", "state")

    def __init__(self):
        self.workspace = self.state = (-1, None)
        self.scalars = (-1, None, None, 0, 0)


def _first_use(kept: dict, handle: int) -> _Kept:
    """For a stream that a layer has not been used on.  A graph is captured on a stream of its own, and uses what the
    layer keeps for the newest of its other streams (that of the warm-up): a state made during the capture would be
    cleared by the graph's replays, at each of them, and by nothing else."""
    if kept and torch.cuda.is_current_stream_capturing():
        return next(reversed(list(kept.values())))
    return kept.setdefault(handle, _Kept())


def _dense_layout(t: Tensor) -> Layout:
    """The layout of a tensor with no halo on its channel and sample dimensions."""
    l = t.layout
    if l.channel_halo:
        raise NotImplementedError("halo on the channel or sample dimension is not supported")
    return l


def _tensor_geometry(l: Layout, num_samples: int):
    """h2x_tensor_geometry of a local tensor (local shape + get_strides()), as something the
    native calls take for a pointer; keep it until the call has returned."""
    if num_samples == l.samples:
        return l.geometry_address
    g = capi.TensorGeometry.from_buffer_copy(l.geometry)
    g.local_shape[g.num_dims - 1] = num_samples
    return _Struct(g)


class _Struct:
    """A ctypes structure as a pointer argument of the native calls."""

    def __init__(self, value):
        self._value = value

    def data_ptr(self) -> int:
        return ctypes.addressof(self._value)


def _share_a_haloed_geometry(l0: Layout, *layouts: Layout) -> bool:
    """Tensors with a halo on a spatial dimension whose local parts lie in memory alike."""
    if not l0.haloed or l0.channel_halo:
        return False
    alike = l0.alike
    for l in layouts:
        if l.alike != alike:
            return False
    return True


def _pair_in_order(l0: Layout, *layouts: Layout) -> bool:
    """Dense tensors: the dense entry points pair the elements of a channel in order whatever the
    extents (4-D and 5-D with one plane, H x W and W x H; the strided ones refuse them), provided
    all have the memory for the samples of `l0`."""
    return l0.dense and all(l.dense and l.samples * l.channels >= l0.samples * l0.channels for l in layouts)


class BatchNormalization:
    """BatchNormalization<Backend, DataType>
    (legacy/include/distconv/dnn_backend/batchnorm.hpp:100-581).

    ``allreduce``, if given, is called as ``allreduce(list_of_per_channel_tensors)``
    where the reference sums over ranks (batchnorm.hpp:185-214,360-400); with the
    default ``None`` the layer is a single rank and the step is the identity.

    Calls on different streams may run at the same time if their outputs are apart.  A captured
    graph shares the buffers of a stream (_first_use): its replays and the calls there follow one another.
    """

    def __init__(self, num_dims: int, decay: float, epsilon: float, global_stats: bool = False,
                 allreduce: Optional[Callable[[List[torch.Tensor]], None]] = None,
                 stream: Optional[torch.cuda.Stream] = None, fuse_local: bool = True,
                 clear_output_halo: bool = False):
        if num_dims not in (4, 5):
            raise ValueError("4-D (NCHW) or 5-D (NCDHW) tensors only")  # batchnorm.cu:259-270
        self.num_dims, self.decay, self.epsilon = num_dims, float(decay), float(epsilon)
        self.global_stats, self.allreduce, self.stream = global_stats, allreduce, stream
        # forward()/backward() of a rank that all-reduces nothing between its two
        # stages run as one or two launches each (h2x_bn_forward_once / _backward_once);
        # the staged methods always use the staged entry points
        self.fuse_local = fuse_local
        # Haloed tensors of one geometry: normalise and the input gradient also clear
        # the halo of their output (what Convolution::forward does to its input before
        # every exchange, convolution.hpp:400-411), in one pass over the real tensors
        # (h2x_bn_batch_normalization_clearing / h2x_bn_backprop2_clearing).  Off by
        # default: the reference's kernels leave halo cells alone.
        self.clear_output_halo = clear_output_halo
        self.num_current_samples = 0
        self._lib = capi.load()
        self._calls = capi.calls()
        self._kept = {}  # by the handle of a stream

    # batchnorm.hpp:467-475
    def set_num_samples(self, n: int) -> None:
        self.num_current_samples = int(n)

    def _ws(self, num_channels: int, st: int) -> torch.Tensor:
        kept = self._kept.get(st) or _first_use(self._kept, st)
        channels, ws = kept.workspace
        if channels != num_channels:
            ws = _buffer_of(self.stream, self._lib.h2x_bn_workspace_bytes(num_channels), torch.uint8)
            kept.workspace = num_channels, ws
        return ws

    def _team_state(self, l: Layout, clearing: bool, st: int) -> Optional[torch.Tensor]:
        """Where the workgroups that share a channel exchange its sums; None where no workgroups do."""
        if l.small_channels:
            return None
        kept = self._kept.get(st) or _first_use(self._kept, st)
        channels, state = kept.state
        if channels < l.channels:
            nbytes = (l.ordered_state_bytes if l.dtype == capi.F64 else
                      l.clearing_team_state_bytes if clearing else l.team_state_bytes)
            if nbytes == 0:
                return None
            state = _buffer_of(self.stream, nbytes, torch.uint8, zero=True)
            kept.state = l.channels, state
        return state

    def _buffers(self, l: Layout, st: int):
        """The workspace and the state of a call, from one look at what is kept for its stream: a small call spends as long on
        looking things up as on anything but the launch."""
        kept = self._kept.get(st) or _first_use(self._kept, st)
        num_channels = l.channels
        channels, ws = kept.workspace
        if channels != num_channels:
            ws = self._ws(num_channels, st)
        if l.small_channels:
            return ws, None
        channels, state = kept.state
        return ws, state if channels >= num_channels else self._team_state(l, False, st)

    @property
    def _state(self) -> Optional[torch.Tensor]:
        """The state for calls on the stream that a call would go to."""
        kept = self._kept.get(_stream_handle(self.stream))
        return kept and kept.state[1]

    def _num_per_sum(self, t: Tensor) -> int:
        """Elements per channel of the global (global_stats) or local shape
        (batchnorm.hpp:232-236,414-418)."""
        return self._elements_per_sum(t.layout)

    # ---- forward -----------------------------------------------------------
    def forward_stage1(self, input: Tensor, mean: torch.Tensor, var: torch.Tensor,
                       is_training: bool = True) -> int:
        lx = input.layout
        self.num_current_samples = lx.samples
        if not is_training:
            return 0
        _dense_layout(input)
        ns, st = lx.samples if lx.active else 0, _stream_handle(self.stream)
        if lx.dense:
            capi.check(self._calls.h2x_bn_channel_sums_and_sqsums(
                lx.dtype, ns, lx.channels, lx.spatial, lx.spatial_real, input, mean, var,
                self._ws(lx.channels, st), st), "channel_sums_and_sqsums")
        else:  # halo on an inner spatial dimension: the generic path of batchnorm.cu:232-248
            capi.check(self._calls.h2x_bn_channel_sums_and_sqsums_strided(
                lx.dtype, ns, _tensor_geometry(lx, ns), input, mean, var,
                self._ws(lx.channels, st), st), "channel_sums_and_sqsums (strided)")
        return 0

    def forward_allreduce(self, mean: torch.Tensor, var: torch.Tensor, is_training: bool = True) -> int:
        if is_training and self.global_stats and self.allreduce is not None:
            self.allreduce([mean, var])
        return 0

    def sums_to_statistics(self, num_per_sum: int, mean, var, running_mean, running_var,
                           dtype: int = capi.F32) -> None:
        """batchnorm.hpp:494-503."""
        capi.check(self._calls.h2x_bn_sums_to_statistics(
            dtype, mean.numel(), num_per_sum, self.decay, mean, var, running_mean, running_var,
            _stream_handle(self.stream)), "sums_to_statistics")

    def batch_normalization(self, input: Tensor, mean, var, scale, bias, output: Tensor) -> None:
        """batchnorm.hpp:505-517."""
        lx, ly = input.layout, output.layout
        if lx.channel_halo or ly.channel_halo:
            _dense_layout(input), _dense_layout(output)  # raises
        ns = self.num_current_samples
        if self.clear_output_halo and ns == lx.samples and _share_a_haloed_geometry(lx, ly):
            capi.check(self._calls.h2x_bn_batch_normalization_clearing(
                lx.dtype, ly.haloed_geometry_address, input.get_buffer(), mean, var, scale, bias,
                output.get_buffer(), self.epsilon, _stream_handle(self.stream)), "batch_normalization (clearing)")
        elif lx.dense and ly.dense:
            status = self._calls.h2x_bn_batch_normalization(
                lx.dtype, ns, lx.channels, lx.spatial, lx.spatial_real, ly.spatial_real, input, mean,
                var, scale, bias, output, self.epsilon, _stream_handle(self.stream))
            if status:
                capi.check(status, "batch_normalization")
        else:
            capi.check(self._calls.h2x_bn_batch_normalization_strided(
                lx.dtype, ns, _tensor_geometry(lx, ns), _tensor_geometry(ly, ns), input, mean, var,
                scale, bias, output, self.epsilon, _stream_handle(self.stream)),
                "batch_normalization (strided)")

    def forward_stage2(self, input: Tensor, mean, var, running_mean, running_var, scale, bias,
                       output: Tensor, is_training: bool = True) -> int:
        if is_training:
            self.sums_to_statistics(self._num_per_sum(input), mean, var, running_mean, running_var,
                                    input.h2x_dtype)
            self.batch_normalization(input, mean, var, scale, bias, output)
        else:
            self.batch_normalization(input, running_mean, running_var, scale, bias, output)  # :243-247
        return 0

    def _elements_per_sum(self, l: Layout) -> int:
        return l.per_channel_global if self.global_stats else l.per_channel_local

    def forward(self, input, mean, var, running_mean, running_var, scale, bias, output,
                is_training: bool = True) -> int:
        lx, ly = input.layout, output.layout
        # (local: no all-reduce between the stages, a rank that owns elements)
        if not is_training:
            # the stages would do nothing but this: no sums, no all-reduce
            self.num_current_samples = lx.samples
            self.batch_normalization(input, running_mean, running_var, scale, bias, output)
            return 0
        local = self.fuse_local and lx.active and (self.allreduce is None or not self.global_stats)
        if local and self.clear_output_halo and (lx.haloed or ly.haloed):
            local = False  # the stages, unless a whole pass clears the halo
            if _share_a_haloed_geometry(lx, ly):
                st = _stream_handle(self.stream)
                status = self._calls.h2x_bn_forward_clearing(
                    lx.dtype, lx.haloed_geometry_address, input.get_buffer(), scale, bias, self._elements_per_sum(lx),
                    self.decay, self.epsilon, mean, var, running_mean, running_var, output.get_buffer(),
                    self._team_state(lx, True, st), st)
                if status != capi.ERR_UNSUPPORTED:
                    self.num_current_samples = lx.samples
                    capi.check(status, "bn forward (clearing)")
                    return 0
        if local:
            if lx.channel_halo or ly.channel_halo:
                _dense_layout(input), _dense_layout(output)  # raises
            ns = self.num_current_samples = lx.samples
            per_sum, st = lx.per_channel_global if self.global_stats else lx.per_channel_local, _stream_handle(self.stream)
            if lx.extents != ly.extents and _pair_in_order(lx, ly):
                capi.check(self._calls.h2x_bn_forward_local(
                    lx.dtype, ns, lx.channels, lx.spatial, lx.spatial_real, ly.spatial_real, input,
                    scale, bias, per_sum, self.decay, self.epsilon, mean, var, running_mean, running_var,
                    output, self._ws(lx.channels, st), st), "bn forward (local)")
                return 0
            ws, state = self._buffers(lx, st)
            status = self._calls.h2x_bn_forward_once(
                lx.dtype, ns, lx.geometry_address, ly.geometry_address if ly.samples == ns else _tensor_geometry(ly, ns),
                input, scale, bias, per_sum, self.decay, self.epsilon, mean, var, running_mean, running_var, output,
                ws, state, st)
            if status:
                capi.check(status, "bn forward (local)")
            return 0
        self.forward_stage1(input, mean, var, is_training)
        self.forward_allreduce(mean, var, is_training)
        return self.forward_stage2(input, mean, var, running_mean, running_var, scale, bias, output,
                                   is_training)

    # ---- backward ----------------------------------------------------------
    def backward_stage1(self, input: Tensor, d_output: Tensor, mean, var, scale, scale_gradient,
                        bias_gradient, mean_gradient, var_gradient) -> int:
        lx, ld = _dense_layout(input), _dense_layout(d_output)
        self.num_current_samples = lx.samples
        ns, st = lx.samples if lx.active else 0, _stream_handle(self.stream)
        tail = (mean, var, scale, scale_gradient, bias_gradient, mean_gradient, var_gradient, self.epsilon,
                self._ws(lx.channels, st), st)
        if lx.dense and ld.dense:
            capi.check(self._calls.h2x_bn_backprop1(
                lx.dtype, ns, lx.channels, lx.spatial, lx.spatial_real, ld.spatial_real, input,
                d_output, *tail), "backprop1")
        else:
            capi.check(self._calls.h2x_bn_backprop1_strided(
                lx.dtype, ns, _tensor_geometry(lx, ns), _tensor_geometry(ld, ns), input,
                d_output, *tail), "backprop1 (strided)")
        return 0

    def backward_allreduce(self, scale_gradient, bias_gradient, mean_gradient, var_gradient,
                           skip_weights: bool = False) -> int:
        if not self.global_stats or self.allreduce is None:  # batchnorm.hpp:367-368
            return 0
        self.allreduce([mean_gradient, var_gradient])
        if not skip_weights:
            self.allreduce([scale_gradient])
            self.allreduce([bias_gradient])
        return 0

    def backward_stage2(self, input: Tensor, d_output: Tensor, mean, var, scale, mean_gradient,
                        var_gradient, d_input: Tensor) -> int:
        lx, ld, li = _dense_layout(input), _dense_layout(d_output), _dense_layout(d_input)
        ns = self.num_current_samples
        tail = (input, d_output, mean, var, scale, mean_gradient, var_gradient,
                d_input, self.epsilon, _stream_handle(self.stream))
        if self.clear_output_halo and ns == lx.samples and _share_a_haloed_geometry(lx, ld, li):
            capi.check(self._calls.h2x_bn_backprop2_clearing(
                lx.dtype, self._num_per_sum(input), li.haloed_geometry_address, input.get_buffer(),
                d_output.get_buffer(), mean, var, scale, mean_gradient, var_gradient, d_input.get_buffer(),
                self.epsilon, _stream_handle(self.stream)), "backprop2 (clearing)")
        # the reference takes its fast path only for halo-free tensors (batchnorm.cu:1503-1506)
        elif lx.dense and ld.dense and li.dense:
            capi.check(self._calls.h2x_bn_backprop2(
                lx.dtype, ns, lx.channels, lx.spatial, lx.spatial_real, ld.spatial_real, li.spatial_real,
                self._num_per_sum(input), *tail), "backprop2")
        else:
            capi.check(self._calls.h2x_bn_backprop2_strided(
                lx.dtype, ns, self._num_per_sum(input), _tensor_geometry(lx, ns), _tensor_geometry(ld, ns),
                _tensor_geometry(li, ns), *tail), "backprop2 (strided)")
        return 0

    def backward(self, input, d_output, mean, var, scale, scale_gradient, bias_gradient,
                 mean_gradient, var_gradient, d_input) -> int:
        lx, ld, li = input.layout, d_output.layout, d_input.layout
        local = self.fuse_local and lx.active and (self.allreduce is None or not self.global_stats)
        if local and self.clear_output_halo and (lx.haloed or ld.haloed or li.haloed):
            local = False
            if _share_a_haloed_geometry(lx, ld, li):
                st = _stream_handle(self.stream)
                status = self._calls.h2x_bn_backward_clearing(
                    lx.dtype, self._elements_per_sum(lx), lx.haloed_geometry_address, input.get_buffer(),
                    d_output.get_buffer(), mean, var, scale, scale_gradient, bias_gradient, mean_gradient,
                    var_gradient, d_input.get_buffer(), self.epsilon, self._team_state(lx, True, st), st)
                if status != capi.ERR_UNSUPPORTED:
                    self.num_current_samples = lx.samples
                    capi.check(status, "bn backward (clearing)")
                    return 0
        if local:
            if lx.channel_halo or ld.channel_halo or li.channel_halo:
                _dense_layout(input), _dense_layout(d_output), _dense_layout(d_input)  # raises
            ns = self.num_current_samples = lx.samples
            per_sum, st = lx.per_channel_global if self.global_stats else lx.per_channel_local, _stream_handle(self.stream)
            if (lx.extents != ld.extents or lx.extents != li.extents) and _pair_in_order(lx, ld, li):
                capi.check(self._calls.h2x_bn_backward_local(
                    lx.dtype, ns, lx.channels, lx.spatial, lx.spatial_real, ld.spatial_real, li.spatial_real, per_sum,
                    input, d_output, mean, var, scale, scale_gradient, bias_gradient,
                    mean_gradient, var_gradient, d_input, self.epsilon, self._ws(lx.channels, st), st),
                    "bn backward (local)")
                return 0
            ws, state = self._buffers(lx, st)
            status = self._calls.h2x_bn_backward_once(
                lx.dtype, ns, per_sum, lx.geometry_address, ld.geometry_address if ld.samples == ns else _tensor_geometry(ld, ns),
                li.geometry_address if li.samples == ns else _tensor_geometry(li, ns),
                input, d_output, mean, var, scale, scale_gradient, bias_gradient,
                mean_gradient, var_gradient, d_input, self.epsilon, ws, state, st)
            if status:
                capi.check(status, "bn backward (local)")
            return 0
        self.backward_stage1(input, d_output, mean, var, scale, scale_gradient, bias_gradient,
                             mean_gradient, var_gradient)
        self.backward_allreduce(scale_gradient, bias_gradient, mean_gradient, var_gradient)
        return self.backward_stage2(input, d_output, mean, var, scale, mean_gradient, var_gradient,
                                    d_input)


def _local_geometry(t: Tensor, region: Optional[Sequence[int]] = None) -> capi.TensorGeometry:
    """Local shape (or a region of it that starts at the first interior element)
    and the strides of the real allocation."""
    g = capi.TensorGeometry()
    nd = t.get_num_dims()
    g.num_dims = nd
    strides = t.get_strides()
    for i in range(nd):
        g.local_shape[i] = t.local_shape[i] if region is None else region[i]
        g.strides[i] = strides[i]
    return g


def transform(op: int, tensors: Sequence[Tensor], params: Sequence[float] = (),
              stream: Optional[torch.cuda.Stream] = None) -> None:
    """tensor::Transform over the interiors of 1-4 tensors of equal local shape
    (legacy/include/distconv/tensor/algorithms/transform_cuda.hpp:359-693) for the
    functors the library names: capi.TRANSFORM_SCALE (t *= p0), TRANSFORM_COPY
    (t1 = t0), TRANSFORM_SCALE_BIAS (t1 = p0 * t0 + p1), TRANSFORM_SUMS_TO_STATISTICS
    (mean, var, running_mean, running_var; p0 = count, p1 = decay)."""
    n = len(tensors)
    for t in tensors:
        if list(t.local_shape) != list(tensors[0].local_shape):
            raise ValueError("tensors of a transform must have the same local shape")  # :383-390
    if tensors[0].get_local_size() == 0:
        return
    gp = (ctypes.c_void_p * n)(*[t.layout.geometry_address for t in tensors])
    tp = (ctypes.c_void_p * n)(*[t.get_base_ptr() for t in tensors])
    pp = (ctypes.c_double * 4)(*(list(params) + [0.0] * (4 - len(params))))
    capi.check(capi.calls().h2x_tensor_transform(op, tensors[0].h2x_dtype, n, ctypes.addressof(gp),
                                                 ctypes.addressof(tp), ctypes.addressof(pp), _stream_handle(stream)),
               "tensor transform")


_reduce_workspaces = {}


def reduce_sum(src: Tensor, dst: Tensor, square: bool = False, region: Optional[Sequence[int]] = None,
               stream: Optional[torch.cuda.Stream] = None) -> None:
    """tensor::ReduceSum / TransformReduceSum (reduce_sum_cuda.hpp:388-439,
    transform_reduce_sum_cuda.hpp:17-87): dst += sum of src (of its squares) over
    every dimension along which dst's local extent is 1.  The sum over ranks that
    the reference ends with (reduce_sum_cuda.hpp:186-192) is the caller's."""
    lib = capi.load()
    gs, gd = _local_geometry(src, region), _local_geometry(dst)
    need = lib.h2x_tensor_reduce_sum_workspace_bytes(ctypes.byref(gs), ctypes.byref(gd))
    key = _stream_handle(stream)
    ws = _reduce_workspaces.get(key)
    if ws is None or ws.numel() < need:
        ws = _reduce_workspaces[key] = _buffer_of(stream, max(need, 256), torch.uint8)
    capi.check(capi.calls().h2x_tensor_reduce_sum(src.h2x_dtype, ctypes.addressof(gs), src.get_base_ptr(),
                                                  ctypes.addressof(gd), dst.get_base_ptr(), int(square), ws, key),
               "tensor reduce_sum")


class SoftmaxMode(Enum):
    """legacy/include/distconv/base.hpp (SoftmaxMode)."""
    INSTANCE = 0
    CHANNEL = 1


class Softmax:
    """Softmax<Backend> (legacy/include/distconv/dnn_backend/softmax.hpp:14-63).

    ``allreduce(values, is_max)``, if given, is called on the per-sample scalars of
    instance mode where the reference all-reduces them over the ranks that share
    a sample (softmax.hpp:52-62); ``None`` means every sample is whole on this rank.

    Calls on different streams and captured graphs: as BatchNormalization's.
    """

    def __init__(self, stream: Optional[torch.cuda.Stream] = None,
                 allreduce: Optional[Callable[[torch.Tensor, bool], None]] = None):
        self.stream, self.allreduce = stream, allreduce
        self.mode = SoftmaxMode.CHANNEL
        self._lib = capi.load()
        self._calls = capi.calls()
        self._kept = {}  # by the handle of a stream

    def setup(self, input: Tensor, mode: SoftmaxMode) -> None:
        self.mode = mode

    @staticmethod
    def _geometry(t: Tensor) -> Layout:
        l = t.layout
        if l.haloed:
            raise NotImplementedError("softmax assumes a dense local tensor")  # softmax.cu:562-563
        return l

    def _buffers(self, l: Layout, t: Tensor, count: int, st: int):
        """The workspace; kept.scalars, whose last two are the addresses of `count` scalars of t's type that nobody reads after
        the call (hold it until then); and where the workgroups that share a sample exchange its partial results (None where
        no workgroups do).  count = 0: the workspace alone.  (In one go, and by what stands beside each buffer: a call for
        each, and to ask the tensors, would be a tenth of a small softmax.)"""
        kept = self._kept.get(st) or _first_use(self._kept, st)
        held, ws = kept.workspace
        need = l.instance_workspace_bytes
        if held < need:
            ws = _buffer_of(self.stream, need, torch.uint8)
            kept.workspace = need, ws
        if count == 0:
            return ws, None, None
        scalars = kept.scalars
        if scalars[0] < count or scalars[1] is not t.dtype:
            buffer = _buffer_of(self.stream, 2 * count, t.dtype)
            address = buffer.data_ptr()
            scalars = kept.scalars = count, t.dtype, buffer, address, address + count * t.dtype.itemsize
        need = l.instance_state_bytes
        if need == 0:
            return ws, scalars, None
        held, state = kept.state
        if held < need:
            state = _buffer_of(self.stream, need, torch.uint8, zero=True)
            kept.state = need, state
        return ws, scalars, state

    def forward(self, x: Tensor, y: Tensor) -> int:
        l = self._geometry(x)
        n = l.samples
        if n == 0:
            return 0
        st = _stream_handle(self.stream)
        if self.mode == SoftmaxMode.CHANNEL:
            status = self._calls.h2x_softmax_channel_forward(
                l.dtype, n, l.channels, l.spatial, x, y, st)
            if status:
                capi.check(status, "softmax forward")
            return 0
        # instance mode: softmax.cu:723-746
        calls, dt, size = self._calls, l.dtype, l.channels * l.spatial
        if self.allreduce is None:
            # every sample is whole on this rank: the stages need not be separate calls
            ws, scalars, state = self._buffers(l, x, n, st)
            status = calls.h2x_softmax_instance_forward_once(
                dt, n, size, x, y, scalars[3], scalars[4], ws, state, -1, st)
            if status:
                capi.check(status, "softmax instance forward")
            return 0
        ws, _, _ = self._buffers(l, x, 0, st)
        smax, sexp = (_buffer_of(self.stream, n, x.dtype, x.device) for _ in range(2))
        capi.check(calls.h2x_softmax_instance_max(dt, n, size, x, smax, ws, st),
                   "softmax instance max")
        self.allreduce(smax, True)
        capi.check(calls.h2x_softmax_instance_exp(dt, n, size, x, smax, y, sexp, ws,
                                                  st), "softmax instance exp")
        self.allreduce(sexp, False)
        capi.check(calls.h2x_softmax_instance_normalize(dt, n, size, sexp, y, st),
                   "softmax instance normalize")
        return 0

    def backward(self, y: Tensor, dy: Tensor, dx: Tensor) -> int:
        l = self._geometry(dx)
        n, dt = l.samples, y.layout.dtype
        if n == 0:
            return 0
        st = _stream_handle(self.stream)
        if self.mode == SoftmaxMode.CHANNEL:
            status = self._calls.h2x_softmax_channel_backward(
                dt, n, l.channels, l.spatial, y, dy, dx, st)
            if status:
                capi.check(status, "softmax backward")
            return 0
        # instance mode: softmax.cu:770-783
        calls, size = self._calls, l.channels * l.spatial
        if self.allreduce is None:
            ws, scalars, state = self._buffers(l, y, n, st)
            status = calls.h2x_softmax_instance_backward_once(
                dt, n, size, y, dy, dx, scalars[3], ws, state, -1, st)
            if status:
                capi.check(status, "softmax instance backward")
            return 0
        ws, _, _ = self._buffers(l, y, 0, st)
        sdp = _buffer_of(self.stream, n, y.dtype, y.device)
        capi.check(calls.h2x_softmax_instance_dot(dt, n, size, y, dy, sdp, ws, st),
                   "softmax instance dot")
        self.allreduce(sdp, False)
        capi.check(calls.h2x_softmax_instance_gradient(dt, n, size, y, dy, sdp,
                                                       dx, st), "softmax instance gradient")
        return 0


class HaloExchangeAccumOp(Enum):
    """legacy/include/distconv/tensor/halo_exchange.hpp:8-9."""
    ID = capi.HALO_ID
    SUM = capi.HALO_SUM
    MAX = capi.HALO_MAX
    MIN = capi.HALO_MIN


# what the launches that serve a whole grid refuse (and then launch nothing) goes through buffers
_NOT_FOR_THE_GRID = (capi.ERR_UNSUPPORTED, capi.ERR_TOO_LARGE)


class HaloExchangeVirtual:
    """HaloExchange for all virtual ranks of one distributed tensor
    (legacy/include/distconv/tensor/halo_exchange_cuda.hpp:18-423).

    The reference object belongs to one rank and hands packed strips to a
    transport.  Here the object holds every rank's local tensor; rank r's send
    buffer for (dim, side) *is* the receive buffer of its neighbour on that
    side for the opposite side, so the transfer is free.  A packed exchange is
    two launches a dimension (pack all ranks and sides, unpack all ranks and
    sides).  A full-width exchange of tensors that share a GPU goes straight
    from tensor to tensor, in one launch (large reverse ones: one a dimension), unless
    a receive buffer was asked for, ``launch_hook`` is set or ``_grid`` names
    another reason.  ``periodic`` wraps neighbours at the grid edge; the reference
    never does (MPI_PROC_NULL, halo_exchange_cuda.hpp:343-345).
    """

    def __init__(self, tensors: Sequence[Tensor], periodic: bool = False,
                 stream: Optional[torch.cuda.Stream] = None):
        self.tensors = list(tensors)
        self.periodic, self.stream = periodic, stream
        self._lib = capi.load()
        self._calls = capi.calls()
        t0 = self.tensors[0]
        self.dist = t0.dist
        if len(self.tensors) != self.dist.num_ranks:
            raise ValueError("one local tensor per rank of the distribution is required")
        if t0.dist.num_ranks != _prod(t0.dist.split_shape):
            raise NotImplementedError("shared (replicated) distributions are not exchanged")  # :30-31
        self.nd = t0.get_num_dims()
        self._recv = {}  # (rank, dim, side) -> torch buffer the rank unpacks from
        self._faces = {}  # exchange arguments and addresses -> launches (label, entry point, descriptors)
        # optional callable(label, launch, num_faces): wraps every launch, for per-kernel timing
        # (of the packing and unpacking launches: a hooked exchange runs dimension by dimension)
        self.launch_hook = None
        self._buffers_wanted = False  # a receive buffer was handed out: exchanges fill them
        # (addresses, is_reverse) of the last exchange that left no strips in the buffers, and the
        # dimensions that were packed after it
        self._direct, self._packed_since = None, ()
        self._grid_of = None  # (addresses, h2x_halo_grid or None, usable for exchanges)

    def get_halo_size(self, rank: int, dim: int, width: int) -> int:
        """halo_exchange_cuda.hpp:267-271."""
        shape = list(self.tensors[rank].local_real_shape)
        shape[dim] = width
        return _prod(shape)

    def is_exchange_required(self, rank: int, dim: int, widths=None) -> bool:
        """halo_exchange_cuda.hpp:305-320."""
        t = self.tensors[rank]
        w = t.overlap[dim] if widths is None else max(widths)
        return self.dist.is_distributed(dim) and self.dist.split_shape[dim] > 1 and w > 0 \
            and t.get_local_size() > 0

    def find_peer_rank(self, rank: int, dim: int, side: int) -> Optional[int]:
        """halo_exchange_cuda.hpp:322-357; None stands for MPI_PROC_NULL."""
        t = self.tensors[rank]
        if not self.is_exchange_required(rank, dim):
            return None
        extent = self.dist.locale_shape[dim]
        p = t.proc_index[dim] + (1 if side == capi.RHS else -1)
        if p < 0 or p >= extent:
            if not self.periodic:
                return None
            p %= extent
        idx = list(t.proc_index)
        idx[dim] = p
        peer = self.dist.rank_of(idx)
        if self.tensors[peer].get_local_size() == 0:
            return None
        return peer

    def _check_widths(self, dim: int, widths) -> None:
        """The receive buffers hold `overlap[dim]` cells per row and the strips lie
        inside the halo: TraverseHalo's precondition, halo_cuda.hpp:909-916."""
        for t in self.tensors:
            if max(widths) > t.overlap[dim]:
                raise ValueError(f"halo width {max(widths)} exceeds the overlap {t.overlap[dim]} of "
                                 f"dimension {dim}")

    def _addresses(self):
        """Device addresses the cached face tables were built for; a tensor that
        was reallocated gets new tables."""
        return tuple([t.data.data_ptr() if t.data is not None else 0 for t in self.tensors])

    def recv_buffer(self, rank: int, dim: int, side: int) -> torch.Tensor:
        """The buffer rank `rank` unpacks its (dim, side) halo from -- and its
        neighbour on that side packs into (get_recv_buffer, halo_exchange_cuda.hpp:277-283).

        Once one has been asked for, every exchange that is not ``fused`` goes through the
        buffers.  An exchange before that may have moved its strips straight from tensor to
        tensor: they are packed now, from the tensors as they are.  That is what was received as
        long as the tensors have not been written since; the cells of a strip that a later dimension's
        phase writes, where strips of two dimensions cross, hold what that phase left."""
        self._buffers_wanted = True
        written = self._direct is not None or (rank, dim, side) not in self._recv
        self._pack_what_was_exchanged()
        buffer = self._receive_buffer(rank, dim, side)
        if written and self.stream is not None and buffer.is_cuda:
            # what the caller does with it on the current stream comes after it was cleared or packed
            torch.cuda.current_stream().wait_stream(self.stream)
        return buffer

    def _pack_what_was_exchanged(self) -> None:
        if self._direct is None:
            return
        addresses, is_reverse = self._direct
        if addresses != self._addresses():
            raise RuntimeError("the tensors were reallocated since the exchange: ask for a receive buffer before it")
        dtype, st = self.tensors[0].h2x_dtype, _stream_handle(self.stream)
        for dim, w in enumerate(self.tensors[0].overlap):
            if dim in self._packed_since:
                continue
            for label, call, arr in self._dim_launches(dim, w, w, w, w, is_reverse, True, HaloExchangeAccumOp.ID, False):
                capi.check(call(dtype, ctypes.addressof(arr), len(arr), st), label)
        self._direct = None

    def _receive_buffer(self, rank: int, dim: int, side: int) -> torch.Tensor:
        key = (rank, dim, side)
        if key not in self._recv:
            t = self.tensors[rank]
            n = self.get_halo_size(rank, dim, t.overlap[dim])  # sized for the full halo (:285-303)
            self._recv[key] = _buffer_of(self.stream, max(n, 1), t.dtype, t.device, zero=True)
        return self._recv[key]

    def make_face(self, rank, dim, side, width, buf, is_pack, is_reverse, op) -> capi.HaloFace:
        """One h2x_halo_face of rank `rank`: what pack_dim / unpack_dim pass down
        (halo_exchange_cuda.hpp:365-393)."""
        t = self.tensors[rank]
        f = capi.HaloFace()
        f.tensor = t.get_buffer()
        f.buffer = buf.data_ptr()
        for i, e in enumerate(t.local_real_shape):
            f.real_shape[i] = e
        f.num_dims, f.dim, f.side, f.width = self.nd, dim, side, width
        f.inner = int((is_pack and not is_reverse) or ((not is_pack) and is_reverse))
        f.is_pack, f.op = int(is_pack), op.value
        return f

    def _grid(self, cells: int) -> int:
        """Address of the h2x_halo_grid of all ranks, or 0 where the launches that serve all of
        them cannot: tensors that do not share a GPU (the packed strips are what could travel),
        ranks that differ in their halo widths or type, an empty rank, a halo on channels or
        samples, or next to a neighbour fewer than `cells` halo widths of interior (an exchange
        needs one: its boundary strips are no halo; a reverse one two: they do not overlap)."""
        kept = self._grid_of
        if kept is None or not self._calls.same_buffers(kept[0], self.tensors):
            kept = self._grid_of = (self._addresses(), *self._make_grid())
        return kept[1] if kept[2] >= cells else 0

    def _make_grid(self):
        """(address of the h2x_halo_grid or 0, halo widths of interior that every rank has)"""
        ts, ov, dtype = self.tensors, self.tensors[0].overlap, self.tensors[0].dtype
        if (any(t.overlap != ov or t.dtype != dtype for t in ts) or len(ts) > capi.HALO_GRID_MAX_RANKS
                or self.nd not in (4, 5) or not any(ov) or any(ov[self.nd - 2:])
                or not _share_a_gpu(ts) or any(not 0 < t.get_local_size() <= t.get_local_real_size() < 2 ** 31 for t in ts)):
            return 0, -1
        ranks = (capi.HaloGridRank * len(ts))()
        cells = 2
        for r, (t, k) in enumerate(zip(ts, ranks)):
            k.tensor = t.get_buffer()
            for d in range(self.nd):
                k.local_shape[d] = t.local_shape[d]
                for side in (capi.LHS, capi.RHS):
                    peer = self.find_peer_rank(r, d, side)
                    k.peer[d][side] = -1 if peer is None else peer
                    if peer is not None:
                        cells = min(cells, t.local_shape[d] // ov[d])
        g = capi.HaloGrid(self.nd, len(ts))
        for d in range(self.nd):
            g.overlap[d] = ov[d]
        g.ranks = ranks
        self._grid_memory = (g, ranks)
        return ctypes.addressof(g), cells

    def exchange_dim(self, dim: int, width_rhs_send: int, width_rhs_recv: int, width_lhs_send: int,
                     width_lhs_recv: int, is_reverse: bool = False, skip_unpack: bool = False,
                     op: HaloExchangeAccumOp = HaloExchangeAccumOp.ID, fused: bool = False) -> None:
        """One dimension for all ranks; the order pack -> (transfer) -> unpack of
        halo_exchange_cuda_mpi.hpp:25-100.  A rank's RHS strip goes to its RHS
        neighbour's LHS receive buffer and vice versa.  With ``fused`` the strips
        move straight from tensor to tensor in one launch (where every rank has at
        least that much interior); the result is the same."""
        if not fused and self._direct is not None and dim not in self._packed_since:
            self._packed_since += (dim,)
        self._issue(self._dim_launches(dim, width_rhs_send, width_rhs_recv, width_lhs_send, width_lhs_recv,
                                       is_reverse, skip_unpack, op, fused))

    def _issue(self, launches) -> None:
        """Launches in order: (label, entry point, array of descriptors)."""
        dtype, st = self.tensors[0].h2x_dtype, _stream_handle(self.stream)
        for label, call, arr in launches:
            if self.launch_hook is None:
                status = call(dtype, ctypes.addressof(arr), len(arr), st)
                if status:
                    capi.check(status, label)
            else:
                self.launch_hook(label, lambda label=label, call=call, arr=arr: capi.check(
                    call(dtype, ctypes.addressof(arr), len(arr), st), label), len(arr))

    def _dim_launches(self, dim, width_rhs_send, width_rhs_recv, width_lhs_send, width_lhs_recv, is_reverse,
                      skip_unpack, op, fused):
        """The launches of one dimension's exchange.  They depend only on the arguments and on
        the tensors' addresses: built once."""
        widths = (width_rhs_send, width_rhs_recv, width_lhs_send, width_lhs_recv)
        self._check_widths(dim, widths)
        if fused and skip_unpack:
            raise ValueError("a fused exchange has no separate unpack to skip")
        key = (dim, widths, is_reverse, skip_unpack, op, fused, self._addresses())
        launches = self._faces.get(key)
        if launches is None:
            # strips of a rank with less than a halo width of interior reach into its halo, which the
            # neighbours' strips are written to: all are read before any is written
            direct = fused and all(t.local_shape[dim] >= max(widths) for t in self.tensors if t.get_local_size())
            build = self._fused_launches if direct else self._staged_launches
            launches = self._faces[key] = build(dim, widths, is_reverse, skip_unpack, op)
        return launches

    def _staged_launches(self, dim, widths, is_reverse, skip_unpack, op):
        width_rhs_send, width_rhs_recv, width_lhs_send, width_lhs_recv = widths
        launches = []
        for group in self._rank_groups(dim, max(widths)):
            packs, unpacks = [], []
            for r in group:
                if not self.is_exchange_required(r, dim, widths):
                    continue
                for side in (capi.LHS, capi.RHS):
                    peer = self.find_peer_rank(r, dim, side)
                    if peer is None:
                        continue
                    w_send = width_rhs_send if side == capi.RHS else width_lhs_send
                    w_recv = width_rhs_recv if side == capi.RHS else width_lhs_recv
                    if w_send > 0:
                        dst = self._receive_buffer(peer, dim, capi.LHS if side == capi.RHS else capi.RHS)
                        packs.append(self.make_face(r, dim, side, w_send, dst, True, is_reverse, op))
                    if w_recv > 0 and not skip_unpack:
                        src = self._receive_buffer(r, dim, side)
                        unpacks.append(self.make_face(r, dim, side, w_recv, src, False, is_reverse, op))
            for what, faces in (("pack", packs), ("unpack", unpacks)):
                if faces:
                    launches.append((f"halo_dim{dim}_{what}", self._calls.h2x_halo_pack_or_unpack_batched,
                                     (capi.HaloFace * len(faces))(*faces)))
        return launches

    def _fused_launches(self, dim, widths, is_reverse, skip_unpack, op):
        # one launch for all ranks: nothing is read back between two launches
        # here, so groups would only add launches (measured: 289 us against 301 us)
        width_rhs_send, width_rhs_recv, width_lhs_send, width_lhs_recv = widths
        moves = []
        for r in range(len(self.tensors)):  # r receives; both of its halos are neighbours in the table
            if not self.is_exchange_required(r, dim, widths):
                continue
            for side in (capi.LHS, capi.RHS):
                peer = self.find_peer_rank(r, dim, side)
                if peer is None:
                    continue
                # what the peer sends towards r leaves the peer on the opposite side
                w_send = width_lhs_send if side == capi.RHS else width_rhs_send
                w_recv = width_rhs_recv if side == capi.RHS else width_lhs_recv
                if w_send != w_recv:
                    raise ValueError("a fused exchange needs equal send and receive widths")
                if w_recv == 0:
                    continue
                src, dst = self.tensors[peer], self.tensors[r]
                m = capi.HaloTransfer()
                m.src, m.dst = src.get_buffer(), dst.get_buffer()
                for i in range(self.nd):
                    m.src_real_shape[i] = src.local_real_shape[i]
                    m.dst_real_shape[i] = dst.local_real_shape[i]
                m.num_dims, m.dim, m.width = self.nd, dim, w_recv
                m.src_side = capi.LHS if side == capi.RHS else capi.RHS
                m.is_reverse, m.op = int(is_reverse), op.value
                moves.append(m)
        if not moves:
            return []
        return [(f"halo_dim{dim}_fused", self._calls.h2x_halo_exchange_fused,
                 (capi.HaloTransfer * len(moves))(*moves))]

    # Faces of the innermost dimension touch one short run per row, and every
    # run costs a whole 128-byte line of memory traffic; the unpack writes into
    # the lines its rank's pack has just read.  Exchanging a few ranks at a time
    # keeps those lines in the 256 MB memory-side cache between the two launches,
    # where the unpack's partial writes merge into whole lines (measured on the
    # 8-rank, 130^3 x 32 case: groups of two ranks, 138 MB of lines, take 275 us,
    # groups of four 290 us, all eight at once more than 300 us).
    _SPARSE_GROUP_BYTES = 160 << 20
    _LINE_BYTES = 128

    def _rank_groups(self, dim: int, width: int) -> List[List[int]]:
        """Partition of the ranks into groups that exchange dimension `dim`
        one after the other.  Neighbours along `dim` always share a group."""
        ranks = list(range(len(self.tensors)))
        t0 = self.tensors[0]
        elem = torch.empty(0, dtype=t0.dtype).element_size()
        if dim != 0 or width * elem >= self._LINE_BYTES:
            return [ranks]
        lines = {}
        for r in ranks:
            idx = list(self.tensors[r].proc_index)
            idx[dim] = 0
            lines.setdefault(tuple(idx), []).append(r)
        groups, current, current_bytes = [], [], 0
        for members in lines.values():
            nbytes = sum(_prod(self.tensors[r].local_real_shape[1:]) * self._LINE_BYTES for r in members)
            if current and current_bytes + nbytes > self._SPARSE_GROUP_BYTES:
                groups.append(current)
                current, current_bytes = [], 0
            current += members
            current_bytes += nbytes
        if current:
            groups.append(current)
        return groups

    def exchange(self, widths_rhs_send=None, widths_rhs_recv=None, widths_lhs_send=None,
                 widths_lhs_recv=None, is_reverse: bool = False, skip_unpack: bool = False,
                 op: HaloExchangeAccumOp = HaloExchangeAccumOp.ID, fused: bool = False) -> None:
        """All dimensions, innermost first, each seeing the halo cells the previous
        ones filled (halo_exchange_cuda.hpp:56-106)."""
        if fused and skip_unpack:
            raise ValueError("a fused exchange has no separate unpack to skip")
        full = widths_rhs_send is widths_rhs_recv is widths_lhs_send is widths_lhs_recv is None
        if (full and (is_reverse or op is HaloExchangeAccumOp.ID) and self.launch_hook is None
                and (fused or not (skip_unpack or self._buffers_wanted))):
            # nobody looks at the receive buffers: straight from tensor to tensor
            grid = self._grid(2 if is_reverse else 1)
            if grid:
                dtype, st = self.tensors[0].h2x_dtype, _stream_handle(self.stream)
                if is_reverse:
                    status = self._calls.h2x_halo_grid_fold(dtype, grid, op.value, st)
                else:
                    status = self._calls.h2x_halo_grid_exchange(dtype, grid, st)
                if status not in _NOT_FOR_THE_GRID:
                    if status:
                        capi.check(status, "halo exchange (grid)")
                    if not fused:
                        self._direct, self._packed_since = (self._grid_of[0], is_reverse), ()
                    return
        ov = self.tensors[0].overlap
        widths = tuple([ov if w is None else w
                        for w in (widths_rhs_send, widths_rhs_recv, widths_lhs_send, widths_lhs_recv)])
        key = ("all", None if full else tuple(map(tuple, widths)), is_reverse, skip_unpack, op, fused, self._addresses())
        launches = self._faces.get(key)
        if launches is None:
            launches = []
            for d in range(self.nd):
                launches += self._dim_launches(d, *(w[d] for w in widths), is_reverse, skip_unpack, op, fused)
            self._faces[key] = launches
        if not fused:
            self._direct = None
        self._issue(launches)

    def clear_halo(self, dim: int) -> None:
        """Tensor::clear_halo (legacy/src/tensor/tensor_mpi_cuda.cu:14-84) on every rank."""
        for t in self.tensors:
            if t.overlap[dim] == 0 or t.get_local_size() == 0:
                continue
            shape = capi.i64_array(t.local_real_shape)
            capi.check(self._calls.h2x_halo_clear(t.h2x_dtype, t.get_buffer(), self.nd, ctypes.addressof(shape),
                                                  dim, t.overlap[dim], _stream_handle(self.stream)), "clear_halo")

    def clear_halos(self, only_unfilled: bool = False) -> None:
        """clear_halo of every dimension that has a halo, on every rank, in batched
        launches: the loop that precedes the forward exchange in Convolution::forward
        (legacy/include/distconv/dnn_backend/convolution.hpp:400-411).

        ``only_unfilled``: only the sides without a neighbour are cleared.  A
        full-width ``exchange()`` that follows overwrites every other halo strip
        completely (a strip spans the whole real extent of the other dimensions);
        the stale values it moves into corner cells on the way are overwritten by a
        later dimension's phase, and a corner that no later phase fills receives
        cleared cells, because neighbours along one dimension sit at the same
        position of every other dimension.  The tensors end up exactly as after
        clearing everything first."""
        grid = self._grid(0)
        if grid:
            status = self._calls.h2x_halo_grid_clear(self.tensors[0].h2x_dtype, grid, int(only_unfilled),
                                                     _stream_handle(self.stream))
            if status not in _NOT_FOR_THE_GRID:
                if status:
                    capi.check(status, "clear_halos (grid)")
                return
        key = ("clear", only_unfilled, self._addresses())
        if key not in self._faces:
            faces = []
            for r, t in enumerate(self.tensors):
                if t.get_local_size() == 0:
                    continue
                for d in range(self.nd):
                    if t.overlap[d] == 0:
                        continue
                    for side in (capi.LHS, capi.RHS):
                        if only_unfilled and self.find_peer_rank(r, d, side) is not None:
                            continue
                        f = capi.HaloFace()
                        f.tensor = t.get_buffer()
                        for i, e in enumerate(t.local_real_shape):
                            f.real_shape[i] = e
                        f.num_dims, f.dim, f.side, f.width, f.inner = self.nd, d, side, t.overlap[d], 0
                        faces.append(f)
            self._faces[key] = (capi.HaloFace * len(faces))(*faces)
        arr = self._faces[key]
        if len(arr):
            capi.check(self._calls.h2x_halo_clear_batched(self.tensors[0].h2x_dtype, ctypes.addressof(arr), len(arr),
                                                          _stream_handle(self.stream)), "clear_halos")


class TensorShufflerVirtual:
    """TensorMPICUDAShuffler for all virtual ranks of a (src, dst) pair of
    distributed tensors (legacy/include/distconv/tensor/shuffle_mpi_cuda.hpp:14-512,
    legacy/src/tensor/shuffle_mpi_cuda.cu:378-476).

    The tables are the reference constructor's (rank_limits per dimension,
    counts and displacements in rank order).  All ranks' receive buffers live in
    one arena and every rank packs straight into its peers' chunks of it -- the
    all-to-all of the reference's ``transfer`` is therefore free -- and each
    direction is two launches: pack for all ranks, unpack for all ranks.

    Tensors that all live on one GPU, no source in a destination's memory, need no
    arena: each direction is one launch from tensor to tensor.  The arenas and the
    packing plans are then never made.
    """

    def __init__(self, src_tensors: Sequence[Tensor], dst_tensors: Sequence[Tensor],
                 stream: Optional[torch.cuda.Stream] = None):
        self.src, self.dst, self.stream = list(src_tensors), list(dst_tensors), stream
        self._lib = capi.load()
        self._calls = capi.calls()
        self._arguments = {}  # addresses of a launch's tensors -> its argument arrays
        if len(self.src) != len(self.dst):
            raise ValueError("source and destination must have the same number of ranks")
        self.num_ranks = len(self.src)
        self.elem_size = torch.empty(0, dtype=self.src[0].dtype).element_size()
        self._directions = {}  # forward? -> plans and buffers of the packed path
        self._direct = None  # (addresses, argument arrays or None): see _direct_arguments
        self._direct_plan = self._make_direct_plan()
        if self._direct_plan is None:
            self._packed(True), self._packed(False)

    @staticmethod
    def get_buf_size(t: Tensor) -> int:
        """shuffle_mpi_cuda.hpp:83-90 (bytes)."""
        return t.get_local_size() * torch.empty(0, dtype=t.dtype).element_size()

    # -- tables (shuffle_mpi_cuda.hpp:129-287) --------------------------------
    @staticmethod
    def rank_limits(a: Tensor, b: Tensor) -> List[int]:
        """End, in a's local coordinates, of each slab of b's process grid."""
        out = []
        for d in range(a.get_num_dims()):
            extent = b.dist.locale_shape[d]
            per = b.dist.get_num_ranks_per_split(d)
            for j in range(extent):
                nxt_root = (j // per + 1) * per  # next split root after j
                nxt = b.get_dimension_rank_offset(d, nxt_root) if nxt_root < extent else b.shape[d]
                lim = 0 if nxt < a.global_index[d] else min(nxt - a.global_index[d], a.local_shape[d])
                out.append(lim)
        return out

    @staticmethod
    def _overlap_size(a: Tensor, b: Tensor, b_index: Sequence[int]) -> int:
        size = 1
        for d in range(a.get_num_dims()):
            b0 = b.get_dimension_rank_offset(d, b_index[d])
            b1 = b0 + b.get_remote_dimension(d, b_index[d])
            lo, hi = max(a.global_index[d], b0), min(a.global_index[d] + a.local_shape[d], b1)
            size *= max(hi - lo, 0)
        return size

    def _counts(self, a: Tensor, b: Tensor) -> List[int]:
        """Elements rank a exchanges with every rank of b's grid, in rank order."""
        counts = []
        for pid in range(self.num_ranks):
            idx = b.dist.rank_index(pid)
            ok = a.is_split_root() and b.dist.is_split_root_index(idx)
            counts.append(self._overlap_size(a, b, idx) if ok else 0)
        return counts

    # -- tensor to tensor -----------------------------------------------------
    def _make_direct_plan(self):
        """Plan of the direct launches, or None where tensors do not share a GPU (packed strips
        are what could travel) or the library cannot express the intersections."""
        tensors, nd = self.src + self.dst, self.src[0].get_num_dims()
        if self.num_ranks > capi.SHUFFLE_DIRECT_MAX_RANKS or not _share_a_gpu(tensors):
            return None
        parts = []
        for ts in (self.src, self.dst):
            arr = (capi.ShufflePart * self.num_ranks)()
            for t, p in zip(ts, arr):
                for d, stride in enumerate(t.get_strides()):
                    p.origin[d], p.extent[d], p.stride[d] = t.global_index[d], t.local_shape[d], stride
                p.active = int(t.is_split_root() and t.get_local_size() > 0)
            parts.append(arr)
        plan = ctypes.c_void_p()
        status = self._lib.h2x_shuffle_direct_plan_create(nd, self.elem_size, self.num_ranks, *parts, ctypes.byref(plan))
        if status in (capi.ERR_UNSUPPORTED, capi.ERR_TOO_LARGE):
            return None
        capi.check(status, "shuffle plan (direct)")
        return plan

    def _direct_arguments(self):
        """Pointer arrays of the direct launches, or None where a source shares memory with a
        destination.  They depend only on the tensors' addresses: kept until one is reallocated."""
        kept = self._direct
        if kept is None or not self._calls.same_buffers(kept[0], self.src, self.dst):
            addresses = tuple([t.data.data_ptr() for t in self.src] + [t.data.data_ptr() for t in self.dst])
            ends = [a + t.data.numel() * self.elem_size for a, t in zip(addresses, self.src + self.dst)]
            n = self.num_ranks
            shared = any(addresses[i] < ends[j] and addresses[j] < ends[i] for i in range(n) for j in range(n, 2 * n))
            arrays = None if shared else tuple(
                (ctypes.c_void_p * n)(*[t.get_base_ptr() for t in ts]) for ts in (self.src, self.dst))
            kept = self._direct = (addresses, arrays, arrays and tuple(ctypes.addressof(a) for a in arrays))
        return kept[2]

    def _shuffle(self, forward: bool) -> None:
        if self._direct_plan is not None:
            args = self._direct_arguments()
            if args is not None:
                status = self._calls.h2x_shuffle_direct(self._direct_plan.value, *args, int(not forward),
                                                        _stream_handle(self.stream))
                if status != capi.ERR_UNSUPPORTED:  # not the device the plan was made on: pack
                    if status:
                        capi.check(status, "shuffle (direct)")
                    return
        d, src, dst = self._packed(forward), *((self.src, self.dst) if forward else (self.dst, self.src))
        self._launch(self._calls.h2x_shuffle_pack_batched, d["pack"], src, d["arena"])
        self._launch(self._calls.h2x_shuffle_unpack_batched, d["unpack"], dst, d["arena"])

    # -- through an arena -----------------------------------------------------
    def _packed(self, forward: bool):
        if forward not in self._directions:
            self._directions[forward] = (self._direction(self.src, self.dst) if forward
                                         else self._direction(self.dst, self.src))
        return self._directions[forward]

    def _direction(self, src: List[Tensor], dst: List[Tensor]):
        """Plans and buffers for src -> dst."""
        n = self.num_ranks
        send_counts = [self._counts(src[r], dst[r]) for r in range(n)]
        recv_counts = [self._counts(dst[r], src[r]) for r in range(n)]
        for r in range(n):
            for p in range(n):
                assert send_counts[r][p] == recv_counts[p][r]
        recv_displs = [[sum(recv_counts[r][:p]) for p in range(n)] for r in range(n)]
        recv_sizes = [sum(recv_counts[r]) for r in range(n)]
        arena_offsets = [sum(recv_sizes[:r]) for r in range(n)]
        arena = _buffer_of(self.stream, max(sum(recv_sizes), 1), src[0].dtype, src[0].device, zero=True)
        if sum(recv_sizes) >= 2 ** 31:
            raise ValueError("arena exceeds the 32-bit displacements of the shuffler tables")
        pack_plans, unpack_plans = [], []
        for r in range(n):
            # pack: chunk for peer p lands in p's receive buffer at the slot reserved for r
            displs = [arena_offsets[p] + recv_displs[p][r] for p in range(n)]
            pack_plans.append(self._plan(src[r], dst[r], self.rank_limits(src[r], dst[r]), displs)
                              if src[r].is_split_root() and src[r].get_local_size() > 0 else None)
            displs = [arena_offsets[r] + recv_displs[r][p] for p in range(n)]
            unpack_plans.append(self._plan(dst[r], src[r], self.rank_limits(dst[r], src[r]), displs)
                                if dst[r].is_split_root() and dst[r].get_local_size() > 0 else None)
        return dict(arena=arena, pack=pack_plans, unpack=unpack_plans,
                    send_counts=send_counts, recv_counts=recv_counts, recv_displs=recv_displs)

    def _plan(self, mine: Tensor, other: Tensor, limits: List[int], displs: List[int]):
        g = capi.ShuffleGeometry()
        g.num_dims, g.elem_size = mine.get_num_dims(), self.elem_size
        for i in range(mine.get_num_dims()):
            g.local_shape[i] = mine.local_shape[i]
            g.strides[i] = mine.get_strides()[i]
            g.peer_locale_shape[i] = other.dist.locale_shape[i]
        rl = (ctypes.c_int32 * len(limits))(*limits)
        dp = (ctypes.c_int32 * len(displs))(*displs)
        g.rank_limits, g.displs = rl, dp
        plan = ctypes.c_void_p()
        capi.check(self._lib.h2x_shuffle_plan_create(ctypes.byref(g), ctypes.byref(plan)),
                   "shuffle plan")
        return plan

    def _launch(self, fn, plans, tensors: List[Tensor], arena: torch.Tensor) -> None:
        live = [t for p, t in zip(plans, tensors) if p is not None]
        if not live:
            return
        n = len(live)
        # the argument arrays depend only on the tensors' addresses: kept until one is reallocated
        addresses = [t.get_base_ptr() for t in live]
        key = (id(fn), id(plans))
        kept = self._arguments.get(key)
        if kept is None or kept[0] != addresses:
            pa = (ctypes.c_void_p * n)(*[p for p in plans if p is not None])
            ta = (ctypes.c_void_p * n)(*addresses)
            ba = (ctypes.c_void_p * n)(*[arena.data_ptr()] * n)
            kept = self._arguments[key] = (addresses, pa, ta, ba)
        _, pa, ta, ba = kept
        capi.check(fn(ctypes.addressof(pa), ctypes.addressof(ta), ctypes.addressof(ba), n,
                      _stream_handle(self.stream)), "shuffle")

    def shuffle_forward(self) -> None:
        """src tensors -> dst tensors (shuffle_mpi_cuda.cu:478-484)."""
        self._shuffle(True)

    def shuffle_backward(self) -> None:
        """dst tensors -> src tensors (shuffle_mpi_cuda.cu:485-490)."""
        self._shuffle(False)

    def __del__(self):
        try:
            for d in self._directions.values():
                for p in d["pack"] + d["unpack"]:
                    if p is not None:
                        self._lib.h2x_shuffle_plan_destroy(p)
            if self._direct_plan is not None:
                self._lib.h2x_shuffle_direct_plan_destroy(self._direct_plan)
        except Exception:
            pass
