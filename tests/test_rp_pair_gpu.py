"""The dedicated wavefronts of the RP launch integrate a bubble on a pair of
lanes, two sub-steps per pass; k_rp_record integrates every bubble of every
launch again on one lane, one sub-step at a time, and compares the sub-step
count and all results bit for bit (frozen-schedule record mode)."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


# one bubble; fewer than a workgroup; one more than a wavefront and a workgroup;
# the last and first population that takes each of the three launches (one bubble
# a wavefront, a queue of lane pairs, a queue of lanes)
@pytest.mark.parametrize("nb", [1, 3, 65, 257, 1024, 1025, 1500, 8192, 8193])
@pytest.mark.parametrize("mixed", [0, 1])
def test_launch_equals_one_lane_integration(brp, nb, mixed):
    prec = brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64
    cfg, b = cases.bubbly_case(64, nb=nb, seed=nb, precision=prec, amp_pa=1.6e6)
    rec = cases.make(brp.Simulation, cfg, b)
    rec.schedule_mode(1)
    s1 = rec.step(130)  # raises where the launch and the record differ
    assert max(s["rp_max_substeps"] for s in s1) > (256 if nb > 3 else 11)
    plain = cases.make(brp.Simulation, cfg, b)
    s2 = plain.step(130)
    assert [s["n_pic"] for s in s1] == [s["n_pic"] for s in s2]
    for n in ("R_t", "R_p", "PG", "Q_B", "sub"):
        np.testing.assert_array_equal(rec.bubbles(n), plain.bubbles(n))
