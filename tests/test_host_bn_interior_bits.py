"""Which elements of a vector are interior ones, in the kernels that clear the halo: every box of small extents, rows shorter than a vector among them,
played on the CPU."""
import itertools

import pytest

from dihydrogen_amd import capi
from test_host_bn_launch_audit import audit_clearing, clearing_geometry


@pytest.mark.parametrize("dtype", [capi.F32, capi.F64])
@pytest.mark.parametrize("width", [1, 2, 3, 4, 5, 8])
def test_vectors_of_small_boxes(width, dtype):
    vectors = 0
    for h, d, lo, hi, beside in itertools.product((1, 2, 3, 4), (None, 1, 2), (0, 1, 2), (0, 1, 3), ((0, 0), (1, 0), (0, 2), (1, 1))):
        if not lo + hi + sum(beside):
            continue
        spatial = (width, h) + (() if d is None else (d,))
        ends = [(lo, hi)] + [beside] * (len(spatial) - 1)
        g = clearing_geometry(spatial, 3, 2, [e[0] for e in ends], [e[1] for e in ends])
        err, rep = audit_clearing(False, dtype, g, [1 << 20, 1 << 30])
        assert err == 0, (spatial, ends)
        launch = rep.launch[0]
        assert all(launch.tensor[t].outside == 0 for t in range(2)), (spatial, ends)
        vectors += launch.vector_width > 1
    assert vectors > 20
