"""The bins a CellManager chooses for its grids (host arithmetic only)."""
import math

import pytest

import pysph_amd.base.api as base
from pysph_amd.base import cell


def _manager(n):
    """A manager of n particles with search radius 1, as far as grids go."""
    cm = base.CellManager(initialize=False)
    cm.cell_size = 1.0
    cm.get_number_of_particles = lambda: n
    return cm


def test_dense_and_sparse_domains():
    # 2 particles a cell in 3D: bins of half the radius; 1 in 100 cells: the
    # reference's cells
    cm = _manager(2 * 50 ** 3)
    assert cm.make_grid((0, 0, 0), (50, 50, 50)).bins_per_cell == 2
    cm = _manager(10000)
    g = cm.make_grid((0, 0, 0), (100, 100, 100))
    assert g.bins_per_cell == 1 and g.cell_size == 1.0
    cm.set_cells_per_radius(3)
    assert cm.make_grid((0, 0, 0), (100, 100, 100)).bins_per_cell == 3


@pytest.mark.parametrize("n,hi", [
    (4 * 10 ** 6, (7e5, 0, 0)),               # 1.4e6 bins along one axis
    (6 * 10 ** 8, (740, 740, 740)),           # 3.3e9 bins in all
])
@pytest.mark.parametrize("at", [0.0, -3e3])
def test_grids_stay_within_their_limits(n, hi, at):
    """Where bins of half the radius would not fit, the grid keeps the
    reference's cells and holds every particle in a cell of its own place."""
    cm = _manager(n)
    lo, hi = (at, 0, 0), (at + hi[0], hi[1], hi[2])
    g = cm.make_grid(lo, hi)
    assert g.bins_per_cell == 1
    for d in range(3):
        assert g.lo[d] <= math.floor(lo[d]) and math.floor(hi[d]) < g.lo[d] + g.dims[d]


@pytest.mark.parametrize("at", [0.6e9, -0.6e9])
def test_cells_far_from_the_origin(at):
    cm = _manager(10 ** 5)
    g = cm.make_grid((at, 0, 0), (at + 100, 0, 0))
    assert g.bins_per_cell == 1
    assert g.lo[0] <= at and at + 100 < g.lo[0] + g.dims[0]
    assert cell.GRID_MAX_OFFSET > abs(at) > cell.GRID_MAX_OFFSET / 2


def test_bounds_around_the_line_keep_the_grid():
    """A sparse set whose bounds swing around the line between one and two
    bins a cell: the grid made first still covers them, with either choice,
    until they are well past the line."""
    n = 1000
    line = cell.CellManager.AUTO_BINS_PER_PARTICLE * n + 32768
    edge = 0.5 * (math.sqrt(line) - 10)          # 2D, 2 (edge + 5) bins an axis
    near, far = 0.97 * edge, 1.03 * edge
    for first, k in ((near, 2), (far, 1)):
        cm = _manager(n)
        cm.grid = cm.make_grid((0, 0, 0), (first, first, 0))
        assert cm.grid.bins_per_cell == k
        for hi in (far, near, far, near):
            # (grown bounds need a larger grid, but not other bins)
            g = cm.make_grid((0, 0, 0), (hi, hi, 0))
            assert g.bins_per_cell == k
            assert cm._covers(cm.grid, g) or hi > first + 1
    cm = _manager(n)
    cm.grid = cm.make_grid((0, 0, 0), (near, near, 0))
    assert cm.make_grid((0, 0, 0), (1.3 * edge, 1.3 * edge, 0)).bins_per_cell == 1
    cm.grid = cm.make_grid((0, 0, 0), (far, far, 0))
    cm.grid.bins_per_cell = 1
    assert cm.make_grid((0, 0, 0), (0.75 * edge, 0.75 * edge, 0)).bins_per_cell == 2
