"""RP launches with more long chains than dedicated wavefronts: the queue's
extreme entries on lane pairs, the others a lane each, and what is left at the
end moved onto pairs, on one workgroup per compute unit and on two.  Every
launch is integrated again one lane and one sub-step at a time and compared
bit for bit (frozen-schedule record mode)."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,lean", [(8201, True), (90001, True), (2000001, False)])
def test_launch_equals_one_lane_integration(brp, nb, lean):
    cfg, b = cases.bubbly_case(64, nb=nb, seed=nb, precision=brp.abi.PREC_MIXED, amp_pa=1.6e6)
    rec = cases.make(brp.Simulation, cfg, b)
    rec.schedule_mode(1)
    s1 = rec.step(125)  # raises where the launch and the record differ
    plain = cases.make(brp.Simulation, cfg, b)
    s2, extreme = [], []
    for _ in range(125):
        s2 += plain.step(1)
        extreme.append(int((plain.bubbles("sub") >= 256).sum()))
    for n in ("R_t", "R_p", "PG", "Q_B", "sub"):
        np.testing.assert_array_equal(rec.bubbles(n), plain.bubbles(n))
    assert [s["rp_max_substeps"] for s in s1] == [s["rp_max_substeps"] for s in s2]
    heavy = [s for s in s2 if s["rp_max_substeps"] >= 512]
    print(nb, "steps with long chains", len(heavy), "lean launches",
          sum(s["rp_lean_launches"] for s in heavy), "of", sum(s["n_pic"] for s in heavy),
          "extreme", max(extreme), flush=True)
    if nb > 8201:  # more than there are dedicated wavefronts; else the tails only
        assert max(extreme) > 256
    # (the first launches of the collapse follow one without long chains)
    assert (2 * sum(s["rp_lean_launches"] for s in heavy) > sum(s["n_pic"] for s in heavy)) == lean
