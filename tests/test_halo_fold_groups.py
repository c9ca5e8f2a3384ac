"""Reverse exchanges of several dimensions in one launch: what is read and written (on the CPU, through the launch audit, which counts a
cell for each of its strips and fails a call in which two threads meet at a cell that one of them stores), and the tensors against the packed
exchange, dimension by dimension, bit for bit."""
import pytest

import test_gpu_direct as direct
import test_host_direct_launch_audit as audits

# (shape, locale grid, overlap), innermost dimension first
GROUPS = [
    ((4, 4, 4, 2, 1), (2, 2, 2, 1, 1), (1, 1, 1, 0, 0)),           # the strips leave nothing of a periodic rank's interior
    ((26, 15, 17, 3, 2), (2, 3, 2, 1, 1), (2, 1, 3, 0, 0)),        # unequal extents and widths, rows with a remainder
    ((13, 140, 31, 2), (3, 2, 1, 1), (1, 1, 0, 0)),                # lines of 5, 4 and 4 cells, 4340 rows: line by line
    ((9, 31, 30, 5, 2), (1, 2, 3, 1, 1), (0, 2, 1, 0, 0)),         # no seam along the rows
    ((12, 9, 20, 2, 1), (2, 1, 4, 1, 1), (1, 0, 2, 0, 0)),         # none along the middle dimension
    ((11, 13, 3, 2), (1, 2, 1, 1), (1, 1, 0, 0)),                  # periodic: a rank is its own neighbour along the rows
    ((60, 64, 62, 4, 1), (2, 2, 2, 1, 1), (1, 1, 1, 0, 0)),        # 8 ranks, some 0.8 MB of strips
]


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("periodic", [False, True])
def test_one_launch_touches_the_strips(periodic, dtype, monkeypatch):
    from dihydrogen_amd import layers
    launches = []

    class Counted(audits.CopyAudit):
        def __exit__(self, *exc):
            result = super().__exit__(*exc)
            launches.append(self.report.launches)
            return result

    monkeypatch.setattr(layers, "_share_a_gpu", lambda tensors: True)
    monkeypatch.setattr(audits, "GRIDS", GROUPS)
    monkeypatch.setattr(audits, "CopyAudit", Counted)
    audits.test_a_grid_of_ranks_touches_the_strips_and_nothing_else("reverse", periodic, dtype)
    assert launches == [1] * len(GROUPS)


def test_large_strips_go_dimension_by_dimension(monkeypatch):
    from dihydrogen_amd import layers
    import torch
    import test_host_copy_launch_audit as packed
    from dihydrogen_amd.layers import HaloExchangeVirtual
    monkeypatch.setattr(layers, "_share_a_gpu", lambda tensors: True)
    for locale, width, launches in (((2, 2, 1, 1), 8, 2), ((2, 2, 1, 1), 4, 1)):  # 0.8 and 0.4 MB of strips
        with audits.CopyAudit() as audit:
            ts = packed._tensors((100, 96, 4, 16), locale, (width, width, 0, 0), torch.float32, audit)
            HaloExchangeVirtual(ts).exchange(is_reverse=True)
        assert audit.report.launches == launches


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("case", GROUPS)
def test_equal_to_the_packed_exchange(case, periodic, dtype):
    direct.test_grid_launches_equal_the_packed_exchange(case, periodic, dtype)
