"""Lists left by a recorded rollout: the end of the recording copies the rows in
use into the context's own buffers, so lists, fields and the next step are the
ones of a run without recording.  One particle, long boundary lists, several
bricks and halos beyond the LDS capacity; exact.
"""
import numpy as np
import pytest

from difffr_amd import scenes
from difffr_amd.simulation import Simulation

pytestmark = pytest.mark.gpu

R = 0.01


@pytest.mark.parametrize("counts,spacing", [((1, 1, 1), 2 * R), ((2, 3, 2), 1.9 * R), ((21, 9, 17), 2 * R),
                                            ((26, 30, 26), 1.72 * R)])
def test_lists_outlive_the_recording(gpu_ready, counts, spacing):
    print(f"[list copy] {counts}", flush=True)
    x = scenes.block_lattice((0.0, 0.0, 0.0), counts, spacing)
    inner = spacing * (np.asarray(counts, np.float64) + 1)
    walls = scenes.box_surface((0.0, 0.0, 0.0), (inner[0], 2.0 * inner[1], inner[2]), 2 * R, open_top=True)
    ball = scenes.sphere_surface(0.03, 2 * R)
    centre = np.array([0.5 * inner[0], x[:, 1].max() + 0.03 + 1.5 * R, 0.5 * inner[2]])
    ident = np.array([1.0, 0, 0, 0])
    sc = scenes.Scene("copy", scenes.default_params(R), x, np.zeros_like(x),
                      [scenes.Body(walls, False, np.zeros(3), ident, 1000.0, name="tank"),
                       scenes.Body(ball, True, centre, ident, 500.0, name="ball")], 2)
    out = []
    for record in (False, True):
        s = Simulation(sc, params_override={"compute_gradient": 0})
        s.set_fixed_iterations([1, 1], [2, 2])
        if record:
            s.adjoint_begin(0)
        s.step(1)
        if record:
            s.adjoint_end()
        r = dict(l0=s.neighbor_lists(0), l1=s.neighbor_lists(1), rho=s.field("density"), alpha=s.field("factor"),
                 s=s.field("sum_grad_p_k"))
        s.step(1)
        r["x"], r["v"] = s.fluid()
        out.append(r)
        s.close()
    a, b = out
    for k in ("l0", "l1"):
        assert len(a[k]) == len(b[k])
        for la, lb in zip(a[k], b[k]):
            np.testing.assert_array_equal(la, lb)
    assert max(len(q) for q in a["l1"]) > 0
    for k in ("rho", "alpha", "s"):
        np.testing.assert_array_equal(a[k], b[k])
    np.testing.assert_allclose(a["x"], b["x"], rtol=0, atol=1e-7)
    np.testing.assert_allclose(a["v"], b["v"], rtol=0, atol=1e-4 * np.abs(a["v"]).max())
