"""The first Picard iteration's RP call is queued before the host knows
whether the step has one: where it has none, nothing may change.  A state
restored to before the wave's arrival makes the first step after it such a
step (the one before it had an iteration)."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


# one bubble a wavefront, a queue of lane pairs, a queue of lanes
@pytest.mark.parametrize("nb", [300, 2000, 9000])
@pytest.mark.parametrize("mixed", [0, 1])
def test_unneeded_call_changes_nothing(brp, nb, mixed):
    cfg, b = cases.bubbly_case(64, nb=nb, seed=3, amp_pa=0.1,
                               precision=brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64)
    fresh = cases.make(brp.Simulation, cfg, b)
    again = cases.make(brp.Simulation, cfg, b)
    again.save_state(0)
    assert again.step(20)[-1]["n_pic"] > 0
    again.restore_state(0)
    for _ in range(8):
        s1, s2 = fresh.step(1)[0], again.step(1)[0]
        assert s1["n_pic"] == s2["n_pic"] and s1["resimax"] == s2["resimax"]
        for n in ("R_t", "R_p", "R_n", "d1R", "PG", "Q_B", "sub", "PL_p", "PL_n", "PL_m", "dt", "re"):
            np.testing.assert_array_equal(again.bubbles(n), fresh.bubbles(n), err_msg=n)
        for n in ("p0", "fg", "fgn", "fgm", "vx"):
            np.testing.assert_array_equal(again.field(n), fresh.field(n), err_msg=n)
        if s1["nstep"] == 1:
            assert s1["n_pic"] == 0
