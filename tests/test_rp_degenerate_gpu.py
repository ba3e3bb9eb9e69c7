"""A bubble whose state no run reaches (a negative radius) is integrated and
flagged like any other, whatever its sub-step count in the step before was: the
first iteration of a step keeps no results."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


# a queue of lane pairs, a queue of lanes
@pytest.mark.parametrize("nb", [2000, 9000])
def test_negative_radius_after_a_long_chain(brp, nb):
    cfg, b = cases.bubbly_case(64, nb=nb, seed=nb, amp_pa=1.6e6)
    cfg.max_substeps = 3000
    a, fresh = (cases.make(brp.Simulation, cfg, b) for _ in range(2))
    a.step(90)
    long = np.zeros(nb, bool)
    for _ in range(60):
        a.step(1)
        long = a.bubbles("sub") >= 256
        if long.any():
            break
    assert long.any()
    # expanding towards zero radius: 2.5 dt v / R = -0.5
    R, v = a.bubbles("R_p"), a.bubbles("d1R")
    v[long] = 0.2 * R[long] / a.info()["dt"]
    R[long] *= -1.0
    a.set_bubble_array("R_p", R)
    a.set_bubble_array("d1R", v)
    fresh.import_state(a.export_state())  # has no sub-step counts
    s, t = a.step(1, check=False)[0], fresh.step(1, check=False)[0]
    print(nb, "long chains", int(long.sum()), "status", s["status"], t["status"], "iterations",
          s["n_pic"], t["n_pic"], flush=True)
    assert s["status"] == t["status"] and s["n_pic"] == t["n_pic"] > 0
    for n in ("R_t", "R_p", "R_n", "d1R", "PG", "Q_B", "sub", "dt", "re"):
        np.testing.assert_array_equal(a.bubbles(n), fresh.bubbles(n), err_msg=n)
