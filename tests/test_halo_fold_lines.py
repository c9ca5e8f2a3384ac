"""Reverse exchanges of thousands of rows, whose innermost dimension goes line of ranks by line of ranks: every
boundary cell folded exactly once (on the CPU, through the launch audit), and the tensors equal the packed
exchange's bit for bit."""
import pytest

import test_gpu_direct as direct
import test_host_direct_launch_audit as audits

# (shape, locale grid, overlap), innermost dimension first; at least 4096 rows a rank unless noted
LINES = [
    ((12, 64, 64, 1), (2, 1, 1, 1), (1, 0, 0, 0)),               # 4096 rows, a pair
    ((12, 63, 65, 1), (2, 1, 1, 1), (1, 0, 0, 0)),               # 4095: rank by rank
    ((13, 22, 100, 2), (3, 1, 1, 1), (2, 0, 0, 0)),              # three ranks of 5, 4 and 4 cells
    ((21, 40, 33, 4), (4, 2, 1, 1), (1, 1, 0, 0)),
    ((35, 50, 31, 3), (5, 1, 1, 1), (3, 2, 0, 0)),               # no whole turns of ranks
    ((9, 20, 22, 5, 5), (2, 2, 2, 1, 1), (2, 1, 3, 0, 0)),       # interiors of 5 and 4 cells, halos of 2
]


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("periodic", [False, True])
def test_every_boundary_cell_is_folded_once(periodic, dtype, monkeypatch):
    from dihydrogen_amd import layers
    monkeypatch.setattr(layers, "_share_a_gpu", lambda tensors: True)
    monkeypatch.setattr(audits, "GRIDS", LINES)
    audits.test_a_grid_of_ranks_touches_the_strips_and_nothing_else("reverse", periodic, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("case", LINES)
def test_equal_to_the_packed_exchange(case, periodic, dtype):
    direct.test_grid_launches_equal_the_packed_exchange(case, periodic, dtype)
