"""Small scenes spread their gather passes (several workgroups a brick, four
lanes a particle) and build their lists a wavefront per cell; larger ones run
one lane per particle.  A scene is run by itself and again with a block of
100,000 particles in free fall well away from it (the grid's corner and so the
bricks stay where they were), which takes the other path at the same pairs.

* lists, fields and velocities after a step: the same bits (the spread passes
  add in the other path's order);
* gradients: the reverse passes add each lane's partial sum at the end.  A sum
  of n FP32 terms is off by at most n x 6e-8 of its terms' magnitudes in either
  order; these scenes' lists hold at most 84 neighbours, fluid and boundary
  together (asserted), so 5e-6, and errors of a few such passes add: 2e-5.

Counts lie at the edges of a wavefront's 16 particles, a workgroup's 160 and the
rules' own limits (44,000 particles in up to 112 filled bricks for the step's
passes, 44,000 and 80,000 for the reverse passes); the compressed block's halos
pass the LDS capacity.
"""
import numpy as np
import pytest

from difffr_amd import scenes
from difffr_amd.simulation import Simulation

pytestmark = pytest.mark.gpu

R = 0.01


def _scene(counts, spacing, far):
    fluid = scenes.block_lattice((0.0, 0.0, 0.0), counts, spacing)
    fluid = fluid + np.random.default_rng(1).uniform(-0.1 * R, 0.1 * R, size=fluid.shape)
    n = fluid.shape[0]
    inner = spacing * (np.asarray(counts, np.float64) + 1)
    walls = scenes.box_surface((0.0, 0.0, 0.0), (inner[0], 2.0 * inner[1], inner[2]), 2 * R, open_top=True)
    ident = np.array([1.0, 0, 0, 0])
    ball = scenes.sphere_surface(0.03, 2 * R)
    centre = np.array([0.5 * inner[0], fluid[:, 1].max() + 0.03 + 1.5 * R, 0.5 * inner[2]])
    bodies = [scenes.Body(walls, False, np.zeros(3), ident, 1000.0, name="tank"),
              scenes.Body(ball, True, centre, ident, 500.0, np.array([0.3, -1.0, 0.2]), np.array([1.0, 0.5, -0.4]),
                          name="ball")]
    if far:
        fluid = np.concatenate([fluid, scenes.block_lattice((inner[0] + 1.0, 0.0, 0.0), (50, 40, 50), 2 * R)])
    vel = np.zeros_like(fluid)
    vel[:n, 1] = 0.5  # towards the ball
    return scenes.Scene("spread", scenes.default_params(R), fluid, vel, bodies, 2), n


@pytest.mark.parametrize("counts,spacing,steps", [
    ((1, 1, 1), 2 * R, 2), ((3, 5, 1), 2 * R, 2), ((4, 4, 1), 1.8 * R, 2), ((17, 1, 1), 1.9 * R, 2),
    ((5, 4, 8), 1.9 * R, 2), ((7, 1, 23), 1.9 * R, 2), ((26, 30, 26), 1.72 * R, 1), ((34, 34, 34), 2 * R, 2),
    ((40, 25, 40), 2 * R, 2), ((40, 30, 35), 1.9 * R, 2), ((42, 30, 35), 1.9 * R, 2), ((43, 43, 43), 2 * R, 2)])
def test_spread_passes_match_one_lane(gpu_ready, counts, spacing, steps):
    seed = np.zeros((2, 7))
    seed[1] = np.random.default_rng(6).normal(size=7)
    out = []
    for far in (False, True):
        sc, n = _scene(counts, spacing, far)
        print(f"[spread] {n} particles, run with {sc.n_fluid}", flush=True)
        s = Simulation(sc, params_override={"compute_gradient": 0})
        s.set_fixed_iterations([1] * steps, [3] * steps)
        s.adjoint_begin(0)
        s.step(1)
        x, v = s.fluid()
        r = {k: s.field(k)[:n] for k in ("density", "factor", "sum_grad_p_k", "density_adv", "kappa", "kappa_v")}
        r.update(x=x[:n], v=v[:n], lists=[s.neighbor_lists(k)[:n] for k in (0, 1)])
        if steps > 1:
            s.step(steps - 1)
        r["grad"] = np.concatenate([s.adjoint_backward(seed)[1], s.adjoint_start_gradient()[1]])
        out.append(r)
        s.close()
    a, b = out
    assert max(len(p) + len(q) for p, q in zip(*a["lists"])) <= 84
    for k in (0, 1):
        for la, lb in zip(a["lists"][k], b["lists"][k]):
            np.testing.assert_array_equal(la, lb)
    for k in ("x", "v", "density", "factor", "sum_grad_p_k", "density_adv", "kappa", "kappa_v"):
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    assert np.abs(a["grad"]).max() > 0.0
    for lo, hi in ((0, 6), (6, 19)):
        scale = np.abs(b["grad"][lo:hi]).max()
        np.testing.assert_allclose(a["grad"][lo:hi], b["grad"][lo:hi], rtol=0, atol=2e-5 * scale)
