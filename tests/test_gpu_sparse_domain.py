"""Little fluid in a large domain: one static sample far away stretches the grid to
a million empty bricks.  The bricks that hold particles keep their cells and their
order, so lists, fields and velocities have the bits of the same scene with that
sample at 0.5 m (out of reach of everything, too), and the gradient agrees within the order of the reverse passes' sums (2e-5,
as derived in test_gpu_spread_passes).
"""
import numpy as np
import pytest

from difffr_amd import scenes
from difffr_amd.simulation import Simulation

pytestmark = pytest.mark.gpu

R = 0.01


def _scene(far):
    x = scenes.block_lattice((0.0, 0.0, 0.0), (10, 10, 10), 1.9 * R)
    x = x + np.random.default_rng(2).uniform(-0.1 * R, 0.1 * R, size=x.shape)
    inner = 1.9 * R * 11.0
    walls = scenes.box_surface((0.0, 0.0, 0.0), (inner, 2.0 * inner, inner), 2 * R, open_top=True)
    ident = np.array([1.0, 0, 0, 0])
    ball = scenes.sphere_surface(0.03, 2 * R)
    centre = np.array([0.5 * inner, x[:, 1].max() + 0.03 + 1.5 * R, 0.5 * inner])
    bodies = [scenes.Body(walls, False, np.zeros(3), ident, 1000.0, name="tank"),
              scenes.Body(ball, True, centre, ident, 500.0, np.array([0.3, -1.0, 0.2]), np.array([1.0, 0.5, -0.4]),
                          name="ball")]
    bodies.append(scenes.Body(np.full((1, 3), far), False, np.zeros(3), ident, 1000.0, name="far"))
    v = np.zeros_like(x)
    v[:, 1] = 0.5
    return scenes.Scene("sparse", scenes.default_params(R), x, v, bodies, 2)


@pytest.mark.parametrize("far", [3.0, 16.5])
def test_far_sample_changes_nothing(gpu_ready, far):
    out = []
    for f in (0.5, far):
        sc = _scene(f)
        print(f"[sparse] far sample at {f}", flush=True)
        seed = np.zeros((len(sc.bodies), 7))
        seed[1] = np.random.default_rng(6).normal(size=7)
        s = Simulation(sc, params_override={"compute_gradient": 0})
        s.set_fixed_iterations([1, 1], [3, 3])
        s.adjoint_begin(0)
        s.step(1)
        r = {k: s.field(k) for k in ("density", "factor", "sum_grad_p_k", "density_adv", "kappa", "kappa_v")}
        r["x"], r["v"] = s.fluid()
        r["lists"] = [s.neighbor_lists(k) for k in (0, 1)]
        s.step(1)
        r["grad"] = s.adjoint_backward(seed)[1]
        out.append(r)
        s.close()
    a, b = out
    for k in (0, 1):
        for la, lb in zip(a["lists"][k], b["lists"][k]):
            np.testing.assert_array_equal(la, lb)
    for k in ("x", "v", "density", "factor", "sum_grad_p_k", "density_adv", "kappa", "kappa_v"):
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    assert np.abs(a["grad"]).max() > 0.0
    np.testing.assert_allclose(a["grad"], b["grad"], rtol=0, atol=2e-5 * np.abs(b["grad"]).max())
