"""Fields come back in particle-id order: what set_field wrote (reordered on the
host) is what field and fluid return (reordered on the device) once the sort has
moved the particles; counts around the reorder's workgroup; exact.
"""
import numpy as np
import pytest

from difffr_amd import native, scenes
from difffr_amd.simulation import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 5000])
def test_fields_in_id_order(gpu_ready, n):
    print(f"[getters] {n}", flush=True)
    rng = np.random.default_rng(n)
    sc = scenes.submerged_body(counts=(20, 16, 20))
    sc.fluid_x = sc.fluid_x[rng.permutation(sc.n_fluid)[:n]]
    sc.fluid_v = np.zeros_like(sc.fluid_x)
    s = Simulation(sc, params_override={"compute_gradient": 0})
    s.step(1)
    x0, _ = s.fluid()
    assert np.abs(x0 - sc.fluid_x).max() < 0.05  # ids kept through the sort
    for name in ("kappa", "kappa_v"):
        w = rng.normal(size=n).astype(np.float32)
        s.set_field(name, w)
        np.testing.assert_array_equal(s.field(name), w)
    x, v = rng.normal(size=(2, n, 3)).astype(np.float32)
    s.set_field("x", x)
    s.set_field("v", v)
    xg, vg = s.fluid()
    np.testing.assert_array_equal(xg, x)
    np.testing.assert_array_equal(vg, v)
    s.close()


def test_error_of_another_call_is_not_the_getters(gpu_ready):
    """An error that some earlier HIP call of the process left (here a device
    number that does not exist) neither fails a getter nor is taken from the
    caller, who may still ask for it."""
    hip = native.load()  # its HIP runtime's functions resolve through it
    s = Simulation(scenes.submerged_body(counts=(6, 5, 6)), params_override={"compute_gradient": 0})
    s.step(1)
    x0, v0 = s.fluid()
    rho = s.field("density")
    hip.hipGetLastError()
    left = hip.hipSetDevice(100000)
    assert left != 0
    x1, v1 = s.fluid()
    np.testing.assert_array_equal(x1, x0)
    np.testing.assert_array_equal(v1, v0)
    np.testing.assert_array_equal(s.field("density"), rho)
    assert hip.hipPeekAtLastError() == left
    hip.hipGetLastError()
    s.close()
