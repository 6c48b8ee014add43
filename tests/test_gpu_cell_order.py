"""The cell sort: every neighbour list runs through the cells in (z, y, x) order
and through a cell in particle-id (sample-index) order, whatever order the
particles arrive in.  Cells of one particle up to most of a list's 64, and a
count beyond one workgroup of the sort; exact.
"""
import numpy as np
import pytest

from difffr_amd import scenes
from difffr_amd.simulation import Simulation

pytestmark = pytest.mark.gpu

R = 0.01
H = 4 * R
CS = H * 1.001


@pytest.mark.parametrize("per_cell,cells", [(1, 1), (2, 1), (16, 1), (17, 2), (60, 1), (9, 64)])
def test_lists_follow_cells_and_ids(gpu_ready, per_cell, cells):
    print(f"[cell order] {cells} cells of {per_cell}", flush=True)
    rng = np.random.default_rng(per_cell)
    side = int(round(cells ** (1 / 3))) if cells > 2 else 1
    grid = np.array([(i % max(side, cells if cells <= 2 else 1), (i // side) % side if side > 1 else 0,
                      i // (side * side) if side > 1 else 0) for i in range(cells)], np.float64)
    walls = scenes.box_surface((0.0, 0.0, 0.0), (8 * CS, 8 * CS, 8 * CS), 2 * R, open_top=True)
    lo = walls.min(0) - 4 * CS
    # cells whose corner is (6, 6, 6) + grid, points off the cells' faces
    x = lo + CS * (6 + np.repeat(grid, per_cell, 0) + rng.uniform(0.01, 0.99, size=(cells * per_cell, 3)))
    x = x[rng.permutation(x.shape[0])].astype(np.float32).astype(np.float64)
    bodies = [scenes.Body(walls, False, np.zeros(3), np.array([1.0, 0, 0, 0]), 1000.0, name="tank")]
    sim = Simulation(scenes.Scene("cells", scenes.default_params(R), x, np.zeros_like(x), bodies, 1))
    sim.set_fixed_iterations([0], [0])
    sim.step(1)
    got, gotb = sim.neighbor_lists(0), sim.neighbor_lists(1)
    sim.close()
    w32 = walls.astype(np.float32).astype(np.float64)

    def expected(p, q, own):
        d2 = np.sum((q - p) ** 2, axis=1)
        near = np.flatnonzero(np.abs(d2 / H ** 2 - 1) < 1e-5)
        assert near.size == 0, "a pair on the support's edge"
        m = np.flatnonzero((d2 < H ** 2) & (np.arange(q.shape[0]) != own))
        c = np.floor((q[m] - lo) / CS).astype(int)
        return m[np.lexsort((m, c[:, 0], c[:, 1], c[:, 2]))]

    for i in range(x.shape[0]):
        np.testing.assert_array_equal(got[i], expected(x[i], x, i))
        wall = np.sort(gotb[i])
        np.testing.assert_array_equal(wall, np.sort(expected(x[i], w32, -1)))
    assert max(len(g) for g in got) >= min(per_cell - 1, 1)
