"""The rigid chain rule (one lane per Jacobian column) against the oracle for
every gradient mode with and without the gyroscopic term and the rotation part,
on two bodies tumbling clear of the fluid: everything is FP64 there, some
hundred operations a step on each side, so 5 steps stay within 5 x 100 x 1.1e-16
of a block's largest entry; held to 1e-12.
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
def test_columns_match_oracle(gpu_ready, mode, gyroscopic, rotation):
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
