"""The rigid chain rule (one lane per Jacobian column) against the oracle for
every gradient mode with and without the gyroscopic term and the rotation part.

* free flight: two bodies tumbling with no fluid in the scene.  No force and no
  per-body sums: the inertia, gyroscopic and quaternion terms by themselves, over
  five steps.  Everything is FP64, some hundred operations a step on each side, so
  5 steps stay within 5 x 100 x 1.1e-16 of a block's largest entry; held to 1e-12.
* coupled: a body in a compressed fluid that closes in on it.  Each step's sums
  and force on the GPU become an affine force law of the oracle (its chain-rule
  hook), which takes one step from the GPU's state and Jacobians before it: all
  eight sums, the force and the torque enter, and nothing but the chain rule is
  compared.  An entry of the result is a sum of some 100 products on three nested
  levels, 100 x 1.1e-16 of their magnitudes; with cancellation up to a hundred
  times, 1e-12 of the block's largest entry.
"""
import numpy as np
import pytest

from difffr_amd import scenes
from difffr_amd.simulation import Simulation
from oracle.pyoracle import OracleSim

pytestmark = pytest.mark.gpu

BLOCKS = [(0, 9), (9, 18), (18, 27), (27, 36), (36, 45), (45, 54), (54, 66), (66, 78)]


@pytest.mark.parametrize("rotation", [0, 1])
@pytest.mark.parametrize("gyroscopic", [0, 1])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_columns_match_oracle_in_free_flight(gpu_ready, mode, gyroscopic, rotation):
    print(f"[chain rule] mode {mode} gyroscopic {gyroscopic} rotation {rotation}", flush=True)
    sc = scenes.submerged_body(body="ellipsoid", counts=(4, 2, 4), steps=5, v0=(0.5, 2.0, 0.2), w0=(9.0, -7.0, 5.0))
    sc.params.update(compute_gradient=1, gradient_mode=mode, gyroscopic=gyroscopic, optimize_rotation=rotation)
    b = sc.bodies[1]
    b.x_rb = b.x_rb + np.array([0.0, 0.5, 0.0])
    x1 = scenes.box_body_surface((0.16, 0.06, 0.1), 0.02)
    sc.bodies.append(scenes.Body(x1, True, b.x_rb + np.array([0.5, 0.1, 0.0]), np.array([0.8, 0.0, 0.6, 0.0]), 700.0,
                                 np.array([-0.2, 1.0, 0.4]), np.array([3.0, 8.0, -6.0]), name="box"))
    g = Simulation(sc)
    o = OracleSim(sc, "f32_rigid64")
    g.step(5)
    o.step(5)
    for k in (1, 2):
        jg, jo = g.jacobians_raw(k), np.asarray(o.jacobians(k)).ravel()
        for lo, hi in BLOCKS:
            scale = max(np.abs(jo[lo:hi]).max(), 1e-3)
            assert np.abs(jg[lo:hi] - jo[lo:hi]).max() <= 1e-12 * scale, (k, lo)
    assert np.abs(jo[45:54] - np.eye(3).ravel()).max() > 1e-4 or not gyroscopic
    g.close()


def _law(net):
    """The sums of a body as the matrices of an affine law in (x, v, omega, q)."""
    m = {n: net[9 * k:9 * k + 9].reshape(3, 3) for k, n in enumerate(("Fv", "Fx", "Fw", "Tw", "Tx", "Tv"))}
    Fq, Tq = net[54:66].reshape(3, 4), net[66:78].reshape(3, 4)
    return np.hstack([m["Fx"], m["Fv"], m["Fw"], Fq]), np.hstack([m["Tx"], m["Tv"], m["Tw"], Tq])


@pytest.mark.parametrize("rotation", [0, 1])
@pytest.mark.parametrize("gyroscopic", [0, 1])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_columns_match_oracle_under_coupling(gpu_ready, mode, gyroscopic, rotation):
    print(f"[chain rule, coupled] mode {mode} gyroscopic {gyroscopic} rotation {rotation}", flush=True)
    sc = scenes.submerged_body(body="ellipsoid", steps=8, v0=(0.5, -0.3, 0.2), w0=(4.0, -3.0, 2.0))
    sc.params.update(compute_gradient=1, gradient_mode=mode, gyroscopic=gyroscopic, optimize_rotation=rotation)
    at = sc.bodies[1].x_rb
    sc.fluid_x[:] = at + 0.93 * (sc.fluid_x - at)
    sc.fluid_v = -0.5 * (sc.fluid_x - at) / 0.07
    g = Simulation(sc)
    dt = float(np.float32(sc.params["dt"]))

    def oracle_step(r, J, net, force, torque):
        o = OracleSim(sc, "f32_rigid64")
        m = o.mass_props(1)["mass"]
        A, B = _law(net)
        o.set_force_model(1, np.zeros(3), np.zeros(3), np.zeros((3, 13)), np.zeros((3, 13)), start=1000)
        o.model_step(3)  # past the release window
        v1 = r["v"] + force * (1.0 / m * dt)
        now = np.concatenate([r["x"], r["v"], r["omega"], r["q"]])
        then = np.concatenate([r["x"] + v1 * dt, v1, r["omega"], r["q"]])
        o.set_force_model(1, force - A @ now, torque - B @ then, A, B, start=2)
        o.set_state("rigid1", np.concatenate([r["x"], r["q"], r["v"], r["omega"]]))
        o.set_state("jac1", J)
        o.model_step(1)
        return np.asarray(o.jacobians(1)).ravel()

    def off(a, b):
        """The largest difference of a block, in units of the block's largest entry."""
        return max(np.abs(a[lo:hi] - b[lo:hi]).max() / max(np.abs(b[lo:hi]).max(), 1e-300) for lo, hi in BLOCKS)

    sharp = 0.0
    g.step(3)
    for _ in range(5):
        r, J = g.rigid(1), g.jacobians_raw(1)
        g.step(1)
        net, after = g.net_gradients_raw(1), g.rigid(1)
        assert min(np.abs(net[lo:hi]).max() for lo, hi in (BLOCKS if rotation else BLOCKS[:2])) > 0.0
        assert np.abs(after["force"]).max() > 0.0 and np.abs(after["torque"]).max() > 0.0
        ours = g.jacobians_raw(1)
        assert off(ours, oracle_step(r, J, net, after["force"], after["torque"])) <= 1e-12
        for lo, hi in BLOCKS if rotation else BLOCKS[:2]:  # the law without one of the sums
            less = net.copy()
            less[lo:hi] = 0.0
            if mode == 0 or (mode == 1 and (lo, hi) in ((0, 9), (18, 27), (27, 36), (45, 54))):
                sharp = off(ours, oracle_step(r, J, less, after["force"], after["torque"]))
                assert sharp > 1e-9, (lo, sharp)
    assert mode == 2 or sharp > 0.0
    g.close()
