"""The cell sort and the list builds: every neighbour list runs through the cells in
(z, y, x) order and through a cell in particle-id (sample-index) order, whatever
order the particles arrive in; exact, order and content, against a direct search.

* cells of one particle up to most of a list's 128 slots, and a count beyond one
  workgroup of the sort, in a corner of three sampled walls: boundary lists with
  more than 64 candidates (the cell-wise build takes 64 a round);
* more than 384 candidates a cell (the cell-wise build keeps six rounds of 64 in
  registers and loads beyond that again for every eight particles) with lists of
  65 to 128, halos within and beyond the LDS capacity, and a cell of more than 32
  particles among them (the items of a cell take eight, and every 32nd from there);
* particles outside the grid, clamped into its border cells.
"""
import numpy as np
import pytest

from difffr_amd import scenes
from difffr_amd.simulation import Simulation

pytestmark = pytest.mark.gpu

R = 0.01
H = 4 * R
H2 = (np.float32(4) * np.float32(R)) * (np.float32(4) * np.float32(R))
CS = H * 1.001
LO = -14.37 * CS  # the grid's corner: four cells before the sample that stretches it


def _bodies():
    """A box of samples off the cells' faces, and one sample far from everything."""
    walls = scenes.box_surface((0.0, 0.0, 0.0), (8 * CS, 8 * CS, 8 * CS), 2 * R, open_top=True)
    x0 = np.concatenate([walls, np.full((1, 3), LO + 4 * CS)])
    return [scenes.Body(x0, False, np.zeros(3), np.array([1.0, 0, 0, 0]), 1000.0, name="tank")]


def _cells(x):
    return np.floor((x - LO) / CS).astype(int)


def _expected(p, q, own, cells):
    """Indices of q's points within the support of p, as the device decides it (FP32, no
    fused operations), by cell and index."""
    d = p.astype(np.float32) - q.astype(np.float32)
    d2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
    m = np.flatnonzero((d2 < H2) & (np.arange(q.shape[0]) != own))
    c = cells[m]
    return m[np.lexsort((m, c[:, 0], c[:, 1], c[:, 2]))]


def _lists(x, start=None):
    """Fluid and boundary lists of a step on x (set after the scene was built on start)."""
    start = x if start is None else start
    sim = Simulation(scenes.Scene("cells", scenes.default_params(R), start, np.zeros_like(x), _bodies(), 1),
                     params_override={"compute_gradient": 0, "max_neighbors": 128})
    if start is not x:
        sim.set_field("x", x)
    sim.set_fixed_iterations([0], [0])
    sim.step(1)
    out = sim.neighbor_lists(0), sim.neighbor_lists(1), sim.halo_stats()
    sim.close()
    return out


def _check(x, got, gotb):
    w = _bodies()[0].x0.astype(np.float32).astype(np.float64)
    c, cw = _cells(x), _cells(w)
    for i in range(x.shape[0]):
        np.testing.assert_array_equal(got[i], _expected(x[i], x, i, c))
        np.testing.assert_array_equal(gotb[i], _expected(x[i], w, -1, cw))


def _candidates(x, q):
    """For each point of x, the points of q in the 27 cells around its own."""
    c, cq = _cells(x), _cells(q)
    return np.array([(np.abs(cq - k).max(1) <= 1).sum() for k in c])


@pytest.mark.parametrize("per_cell,cells", [(1, 1), (2, 1), (16, 1), (17, 2), (60, 1), (9, 64)])
def test_lists_follow_cells_and_ids(gpu_ready, per_cell, cells):
    print(f"[cell order] {cells} cells of {per_cell}", flush=True)
    rng = np.random.default_rng(per_cell)
    side = int(round(cells ** (1 / 3))) if cells > 2 else 1
    grid = np.array([(i % max(side, cells if cells <= 2 else 1), (i // side) % side if side > 1 else 0,
                      i // (side * side) if side > 1 else 0) for i in range(cells)], np.float64)
    # cells next to the one of the walls' corner, points off the cells' faces
    x = LO + CS * (15 + np.repeat(grid, per_cell, 0) + rng.uniform(0.01, 0.99, size=(cells * per_cell, 3)))
    x = x[rng.permutation(x.shape[0])].astype(np.float32).astype(np.float64)
    got, gotb, _ = _lists(x)
    _check(x, got, gotb)
    assert max(len(g) for g in got) >= min(per_cell - 1, 8)
    assert max(len(g) for g in gotb) > 4 or per_cell < 16
    assert _candidates(x, _bodies()[0].x0).max() > 64


@pytest.mark.parametrize("kind", ["block", "large block", "full cell"])
def test_lists_of_crowded_cells(gpu_ready, kind):
    print(f"[cell order] {kind}", flush=True)
    rng = np.random.default_rng(11)
    n, spacing = {"block": (9, 1.45 * R), "large block": (16, 1.45 * R), "full cell": (10, 1.6 * R)}[kind]
    x = LO + 15.0 * CS + scenes.block_lattice((0.0, 0.0, 0.0), (n, n, n), spacing)
    x = x + rng.uniform(-0.1 * R, 0.1 * R, size=x.shape)
    if kind == "full cell":  # the block's middle cell holds 50 particles
        mid = _cells(x.mean(0, keepdims=True))[0]
        x = x[(_cells(x) != mid).any(1)]
        x = np.concatenate([x, LO + CS * (mid + rng.uniform(0.01, 0.99, size=(50, 3)))])
    x = x[rng.permutation(x.shape[0])].astype(np.float32).astype(np.float64)
    got, gotb, halo = _lists(x)
    assert _candidates(x, x).max() > 384
    assert 65 <= max(len(g) for g in got) <= 128
    assert (halo["largest_halo"] > halo["max_capacity"]) == (kind == "large block")
    _check(x, got, gotb)


@pytest.mark.parametrize("axis,side", [(0, 1), (1, 1), (2, -1)])
def test_lists_outside_the_grid(gpu_ready, axis, side):
    print(f"[cell order] outside along {axis} {side}", flush=True)
    rng = np.random.default_rng(5)
    x = LO + CS * (16 + rng.uniform(0.01, 2.99, size=(300, 3)))
    start = x.copy()
    x[:200, axis] += side * 60 * CS  # a cloud of 200 beyond the border, 100 stay
    x = x[rng.permutation(300)].astype(np.float32).astype(np.float64)
    got, _, _ = _lists(x, start)
    c = _cells(x)
    c[np.abs(x[:, axis] - (LO + 17 * CS)) > 30 * CS, axis] = 0  # all in the border cells of that axis
    for i in range(300):
        np.testing.assert_array_equal(got[i], _expected(x[i], x, i, c))
    assert max(len(got[i]) for i in range(300) if abs(x[i, axis] - (LO + 17 * CS)) > 30 * CS) > 8
