"""Performance cases: the calls a program that trains or serves spatially decomposed networks
makes through the layer API (batch-norm, softmax, halo exchange, tensor shuffle), each with the
inputs it has in hand before the call.

Shapes are written N, C, [D,] H, W here; the library's own order is innermost first.
"""
import math

import torch

from dihydrogen_amd import capi
from dihydrogen_amd.layers import (BatchNormalization, HaloExchangeAccumOp, HaloExchangeVirtual, Softmax, SoftmaxMode,
                                   TensorShufflerVirtual)
from dihydrogen_amd.tensor import Distribution, LocaleVirtual, Tensor

_DTYPES = {"float32": torch.float32, "float64": torch.float64}


def _bn(name, n, c, d, h, w, halo=0, dtype="float32", mode="train", clear=False):
    """d = 0: a 4-D tensor.  halo: width on every spatial dimension (a shard of a spatial decomposition)."""
    return {"name": name, "kind": "batchnorm", "n": n, "c": c, "d": d, "h": h, "w": w, "halo": halo, "dtype": dtype,
            "mode": mode, "clear": clear}


def _softmax(name, n, c, h, w, mode="channel", dtype="float32"):
    return {"name": name, "kind": "softmax", "n": n, "c": c, "h": h, "w": w, "mode": mode, "dtype": dtype}


def _halo(name, n, c, d, h, w, gd, gh, gw, width=1, periodic=False, step="forward", fused=False, dtype="float32"):
    """Global extents and the grid of ranks over them."""
    return {"name": name, "kind": "halo", "n": n, "c": c, "d": d, "h": h, "w": w, "gd": gd, "gh": gh, "gw": gw,
            "width": width, "periodic": periodic, "step": step, "fused": fused, "dtype": dtype}


def _shuffle(name, n, c, h, w, ranks, gh, gw, halo=0, dtype="float32"):
    return {"name": name, "kind": "shuffle", "n": n, "c": c, "h": h, "w": w, "ranks": ranks, "gh": gh, "gw": gw,
            "halo": halo, "dtype": dtype}


def listed():
    return [
        # A training step's batch-norm, forward + backward, on an early 2-D activation of a small batch.
        _bn("bn_train_2d_56", 8, 64, 0, 56, 56),
        # The same layer when serving one image: the smallest call, normalisation with running statistics.
        _bn("bn_infer_one_image", 1, 64, 0, 112, 112, mode="infer"),
        # Late activations of a large batch: segments of 49 elements.
        _bn("bn_train_7x7", 128, 1024, 0, 7, 7),
        # Volumetric network, first layers: the largest batch-norm.
        _bn("bn_train_3d_64", 4, 64, 64, 64, 64),
        # One rank's shard of a volumetric network split over three dimensions: haloed rows of an even, unaligned length.
        _bn("bn_train_3d_shard", 8, 64, 30, 30, 30, halo=1),
        # Double precision (validation runs, scientific inputs) on odd extents: nothing is a whole vector.
        _bn("bn_train_3d_odd_f64", 8, 32, 33, 33, 33, dtype="float64"),
        # Segmentation head: softmax over the channels of every pixel, forward + backward.
        _softmax("softmax_pixels_21", 16, 21, 256, 256),
        # More classes than one thread holds, ragged pixel count (a cropped image).
        _softmax("softmax_pixels_150", 4, 150, 65, 97),
        # Classifier: softmax over a whole sample, forward + backward; bound by latency.
        _softmax("softmax_classes_1000", 256, 1000, 1, 1, mode="instance"),
        # Forward halo exchange of a volumetric layer, eight ranks of 128^3.
        _halo("halo_3d_128", 1, 32, 256, 256, 256, 2, 2, 2, periodic=True),
        # What a convolution does before it reads its input: clear what no neighbour fills, exchange; small
        # ragged shards of a 2-D layer on an open 2 x 2 grid.
        _halo("halo_2d_conv_input", 4, 64, 0, 57, 57, 1, 2, 2, step="clear_forward"),
        # Sample-parallel to spatial-parallel and back.
        _shuffle("shuffle_128", 32, 64, 128, 128, 4, 2, 2),
    ]


# No drawn case moves more than the largest listed one (the 3-D batch-norm, 67 million elements five times over).
_MOST_BYTES = 5 * 4 * 67_108_864
_MOST_HALO_ROWS = 8 * 130 * 130 * 32  # innermost rows of all ranks: what an exchange's cost goes with


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _extents(rng, count, lo, hi):
    """Spatial extents of one size, none more than about twice another."""
    size = _log(rng, lo, hi)
    return [min(hi, max(lo, round(size * rng.uniform(0.7, 1.4)))) for _ in range(count)]


def _draw_bn(rng):
    dtype = "float64" if rng.random() < 0.2 else "float32"
    item = 8 if dtype == "float64" else 4
    halo = rng.choice([1, 1, 2]) if rng.random() < 0.35 else 0
    three_d = rng.random() < 0.5
    most = _MOST_BYTES // (5 * item)
    while True:
        if three_d:
            d, h, w = _extents(rng, 3, 4, 96)
            c = _log(rng, 4, 512)
        else:
            d, (h, w) = 0, _extents(rng, 2, 4 if halo else 1, 224)
            c = _log(rng, 8, 2048)
        n = _log(rng, 1, 256)
        elems = n * c * max(d, 1) * h * w
        if 100_000 <= elems <= most and n * max(d, 1) * h * w > 1:
            break
    mode = "infer" if rng.random() < 0.25 else "train"
    return _bn("", n, c, d, h, w, halo, dtype, mode, clear=bool(halo and rng.random() < 0.4))


def _draw_softmax(rng):
    dtype = "float64" if rng.random() < 0.15 else "float32"
    if rng.random() < 0.4:
        return _softmax("", _log(rng, 16, 4096), _log(rng, 10, 4096), 1, 1, rng.choice(["instance", "channel"]), dtype)
    while True:
        n, c, (h, w) = _log(rng, 1, 32), _log(rng, 2, 512), _extents(rng, 2, 7, 384)
        if 50_000 <= n * c * h * w <= 22_020_096:
            return _softmax("", n, c, h, w, "instance" if rng.random() < 0.25 else "channel", dtype)


def _draw_halo(rng):
    three_d = rng.random() < 0.6
    step = rng.choice(["forward", "forward", "clear_forward", "reverse"])
    while True:
        g = [rng.choice([1, 2, 2, 4]) for _ in range(3 if three_d else 2)]
        if not 2 <= math.prod(g) <= 8:
            continue
        ext = [k * e + rng.randrange(k) for k, e in zip(g, _extents(rng, len(g), 6, 128))]
        c, n = _log(rng, 1, 128), _log(rng, 1, 16)
        width = rng.choice([1, 1, 1, 2, 3])
        rows = n * c * math.prod(ext[:-1]) * g[-1]
        cells = n * c * math.prod(ext)
        if cells <= 100_000_000 and rows <= _MOST_HALO_ROWS // 2 and cells >= 20_000:
            break
    d, gd = (ext[0], g[0]) if three_d else (0, 1)
    return _halo("", n, c, d, ext[-2], ext[-1], gd, g[-2], g[-1], width, rng.random() < 0.5, step, rng.random() < 0.4,
                 "float64" if rng.random() < 0.15 else "float32")


def _draw_shuffle(rng):
    while True:
        gh, gw = rng.choice([(2, 1), (2, 2), (4, 1), (4, 2), (1, 2), (4, 4)])
        ranks = gh * gw
        n, c = ranks * _log(rng, 1, 8) + rng.choice([0, 0, 1]), _log(rng, 1, 256)
        h, w = _extents(rng, 2, 16, 256)
        if 100_000 <= n * c * h * w <= 33_554_432:
            break
    return _shuffle("", n, c, h, w, ranks, gh, gw, rng.choice([0, 0, 1]), "float64" if rng.random() < 0.15 else "float32")


def draw(rng):
    kind = rng.choice(["bn", "bn", "bn", "softmax", "softmax", "halo", "halo", "shuffle"])
    case = {"bn": _draw_bn, "softmax": _draw_softmax, "halo": _draw_halo, "shuffle": _draw_shuffle}[kind](rng)
    del case["name"]
    return case


# ---- inputs ------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _prepare_bn(case, seed):
    g, dtype = _generator(seed), _DTYPES[case["dtype"]]
    spatial = [case["w"], case["h"]] + ([case["d"]] if case["d"] else [])
    ns, c = len(spatial), case["c"]
    if case["halo"]:
        # one rank's shard of a tensor split in two along every spatial dimension
        dist = Distribution.make_overlapped_distribution([2] * ns + [1, 1], [case["halo"]] * ns + [0, 0])
        shape, locale = [2 * e for e in spatial] + [c, case["n"]], LocaleVirtual(0, 2 ** ns)
    else:
        dist, shape, locale = Distribution.make_localized_distribution(ns + 2), spatial + [c, case["n"]], LocaleVirtual(0, 1)
    train = case["mode"] == "train"
    x, y = (Tensor(shape, locale, dist, dtype).allocate() for _ in range(2))
    x.interior_view().normal_(0, 1, generator=g)
    vec = lambda: torch.empty(c, dtype=dtype, device="cuda")
    state = {"kind": "batchnorm", "train": train, "x": x, "y": y, "scale": vec().uniform_(0.5, 1.5, generator=g),
             "bias": vec().normal_(0, 0.1, generator=g), "mean": vec().zero_(), "var": vec().fill_(1),
             "running_mean": vec().normal_(0, 0.1, generator=g), "running_var": vec().uniform_(0.5, 1.5, generator=g),
             "layer": BatchNormalization(ns + 2, 0.9, 1e-5, clear_output_halo=case["clear"])}
    state["layer"].set_num_samples(case["n"])
    if train:
        dy, dx = (Tensor(shape, locale, dist, dtype).allocate() for _ in range(2))
        dy.interior_view().normal_(0, 1, generator=g)
        state.update(dy=dy, dx=dx, grads=[vec().zero_() for _ in range(4)])
    return state


def _run_bn(s):
    s["layer"].forward(s["x"], s["mean"], s["var"], s["running_mean"], s["running_var"], s["scale"], s["bias"], s["y"],
                       s["train"])
    if not s["train"]:
        return s["y"].data
    s["layer"].backward(s["x"], s["dy"], s["mean"], s["var"], s["scale"], *s["grads"], s["dx"])
    return [s["y"].data, s["mean"], s["var"], s["running_mean"], s["running_var"], s["dx"].data] + s["grads"]


def _prepare_softmax(case, seed):
    g, dtype = _generator(seed), _DTYPES[case["dtype"]]
    dist = Distribution.make_localized_distribution(4)
    make = lambda: Tensor([case["w"], case["h"], case["c"], case["n"]], LocaleVirtual(0, 1), dist, dtype).allocate()
    s = {"kind": "softmax", "x": make(), "y": make(), "dy": make(), "dx": make(), "layer": Softmax()}
    s["x"].data.normal_(0, 2, generator=g)
    s["dy"].data.normal_(0, 1, generator=g)
    s["layer"].setup(s["x"], SoftmaxMode.INSTANCE if case["mode"] == "instance" else SoftmaxMode.CHANNEL)
    return s


def _run_softmax(s):
    s["layer"].forward(s["x"], s["y"])
    s["layer"].backward(s["y"], s["dy"], s["dx"])
    return s["y"].data, s["dx"].data


def _halo_shape(case):
    """(global shape, grid, halo widths), innermost first."""
    three = [case["d"]] if case["d"] else []
    grid = [case["gw"], case["gh"]] + ([case["gd"]] if three else [])
    shape = [case["w"], case["h"]] + three + [case["c"], case["n"]]
    return shape, grid + [1, 1], [case["width"]] * len(grid) + [0, 0]


def _prepare_halo(case, seed):
    g = _generator(seed)
    shape, grid, widths = _halo_shape(case)
    dist = Distribution.make_overlapped_distribution(grid, widths)
    ranks = [Tensor(shape, LocaleVirtual(r, dist.num_ranks), dist, _DTYPES[case["dtype"]]).allocate()
             for r in range(dist.num_ranks)]
    for t in ranks:
        # a reverse exchange sends gradients that a kernel has left in the halo
        (t.data if case["step"] == "reverse" else t.interior_view()).uniform_(-1, 1, generator=g)
    return {"kind": "halo", "ranks": ranks, "step": case["step"], "fused": case["fused"],
            "exchange": HaloExchangeVirtual(ranks, periodic=case["periodic"])}


def _run_halo(s):
    if s["step"] == "reverse":
        s["exchange"].exchange(is_reverse=True, op=HaloExchangeAccumOp.SUM, fused=s["fused"])
    else:
        if s["step"] == "clear_forward":
            s["exchange"].clear_halos(only_unfilled=True)
        s["exchange"].exchange(fused=s["fused"])
    return [t.data for t in s["ranks"]]


def _prepare_shuffle(case, seed):
    g, dtype, ranks = _generator(seed), _DTYPES[case["dtype"]], case["ranks"]
    shape = [case["w"], case["h"], case["c"], case["n"]]
    src_dist = Distribution([1, 1, 1, ranks])
    grid = [case["gw"], case["gh"], 1, 1]
    dst_dist = (Distribution.make_overlapped_distribution(grid, [case["halo"]] * 2 + [0, 0]) if case["halo"]
                else Distribution(grid))
    src, dst = ([Tensor(shape, LocaleVirtual(r, ranks), dist, dtype).allocate() for r in range(ranks)]
                for dist in (src_dist, dst_dist))
    for t in src:
        t.data.uniform_(-1, 1, generator=g)
    return {"kind": "shuffle", "src": src, "dst": dst, "shuffler": TensorShufflerVirtual(src, dst)}


def _run_shuffle(s):
    s["shuffler"].shuffle_forward()
    s["shuffler"].shuffle_backward()
    return [t.data for t in s["dst"]] + [t.data for t in s["src"]]


_PREPARE = {"batchnorm": _prepare_bn, "softmax": _prepare_softmax, "halo": _prepare_halo, "shuffle": _prepare_shuffle}
_RUN = {"batchnorm": _run_bn, "softmax": _run_softmax, "halo": _run_halo, "shuffle": _run_shuffle}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


# ---- what a pass cannot do without ----------------------------------------------------------------

def _halo_cells(case):
    """Halo cells that receive a neighbour's values, over all ranks, and cells that are cleared."""
    shape, grid, widths = _halo_shape(case)
    dist = Distribution.make_overlapped_distribution(grid, widths)
    filled = cleared = 0
    for r in range(dist.num_ranks):
        t = Tensor(shape, LocaleVirtual(r, dist.num_ranks), dist)
        for d, o in enumerate(t.overlap):
            if not o:
                continue
            strip = t.get_local_real_size() // t.local_real_shape[d] * o
            edges = (t.proc_index[d] == 0) + (t.proc_index[d] == grid[d] - 1)
            open_sides = 0 if case["periodic"] else edges
            filled += (2 - open_sides) * strip
            cleared += open_sides * strip
    return filled, cleared if case["step"] == "clear_forward" else 0


def work(case):
    item = 8 if case["dtype"] == "float64" else 4
    if case["kind"] == "halo":
        filled, cleared = _halo_cells(case)
        # each cell is read where it comes from and written where it goes; a sum also reads its target
        reverse = case["step"] == "reverse"
        return {"bytes": ((3 if reverse else 2) * filled + cleared) * item, "flops": filled if reverse else 0}
    elems = case["n"] * case["c"] * max(case.get("d", 0), 1) * case["h"] * case["w"]
    if case["kind"] == "shuffle":
        return {"bytes": 4 * elems * item, "flops": 0}  # each way: every element read and written
    if case["kind"] == "softmax":
        # forward x -> y, backward y, dy -> dx
        return {"bytes": 5 * elems * item, "flops": 9 * elems}
    if case["mode"] == "infer":
        return {"bytes": 2 * elems * item, "flops": 3 * elems}
    # forward x -> y, backward x, dy -> dx
    return {"bytes": 5 * elems * item, "flops": 24 * elems}


def tolerance(case):
    if case["kind"] == "shuffle" or (case["kind"] == "halo" and case["step"] != "reverse"):
        return "exact"  # copies
    if case["kind"] == "halo":
        # one rounding per strip that is added in, in the data's type
        return {"rel": 1e-6 if case["dtype"] == "float32" else 1e-14}
    # sums over a channel or a pixel's classes, then a few operations in the data's type
    return {"rel": 1e-5 if case["dtype"] == "float32" else 1e-12}
