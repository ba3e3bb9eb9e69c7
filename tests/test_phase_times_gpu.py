"""Phase times are times of the kernels, without the waits for the host that
lie between launches queued before and after a report."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


# one bubble a wavefront, a queue of lanes
@pytest.mark.parametrize("nb", [200, 9000])
def test_motion_queued_ahead_costs_what_it_costs_otherwise(brp, nb):
    cfg, b = cases.bubbly_case(64, nb=nb, seed=3, amp_pa=0.1e6)
    steps = 200
    with cases.make(brp.Simulation, cfg, b) as sim:
        sim.step(120)
        sim.save_state(0)
        one = []
        for _ in range(steps):  # never ahead of the report
            n_pic = sim.step(1)[0]["n_pic"]
            one.append(sim.phase_times()["motion"])
        assert n_pic > 0
        sim.restore_state(0)
        sim.step(steps)
        many = sim.phase_times()["motion"] / steps
    print(nb, "motion, us a step: one at a time", 1e3 * np.median(one), "together", 1e3 * many, flush=True)
    assert many < 1.2 * np.median(one)


# the first RP call is queued ahead of the report in a step after one that had
# an iteration, cylindrical: with the fold at the axis behind it
@pytest.mark.parametrize("nb", [200, 9000])
@pytest.mark.parametrize("cyl", [0, 1])
def test_rp_queued_ahead_costs_what_it_costs_otherwise(brp, nb, cyl):
    cfg, b = cases.bubbly_case(64, nb=nb, seed=3, amp_pa=0.1e6)
    cfg.tr_cylindrical = cyl
    with cases.make(brp.Simulation, cfg, b) as sim:
        sim.save_state(0)  # steps without an iteration
        sim.step(120)
        sim.save_state(1)
        ms = {}
        for after in (0, 1):
            v = []
            for _ in range(100):
                sim.restore_state(after)
                assert (sim.step(1)[0]["n_pic"] > 0) == (after == 1)
                sim.restore_state(1)
                n_pic = sim.step(1)[0]["n_pic"]
                v.append(sim.phase_times()["bubble_rp"] / n_pic)
            ms[after] = np.median(v)
    print(nb, cyl, "RP, us a launch: behind the report", 1e3 * ms[0], "ahead", 1e3 * ms[1], flush=True)
    assert ms[1] < 1.2 * ms[0]
