"""Steps with bubbles that fail: the launches of the next step queued before
the report must leave the failed step's state.  Steps in one call (queued
ahead) against one call a step (never), to the same error, with the same
stats, fields and bubbles."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

BUBBLES = ("x", "y", "vx", "vy", "R_t", "R_p", "R_n", "d1R", "PG", "Q_B", "PL_p", "PL_n", "PL_m",
           "sub", "dt", "re")
FIELDS = ("p0", "px", "py", "vx", "vy", "fg", "fgn", "fgm")


def run(brp, cfg, b, together, poke):
    with cases.make(brp.Simulation, cfg, b) as sim:
        stats = []
        if poke:
            sim.step(70)
            v = sim.bubbles(poke)
            v[0] = 1e305
            sim.set_bubble_array(poke, v)
        while not stats or stats[-1]["status"] == 0:
            assert len(stats) < 200
            stats += [s for s in sim.step(200 if together else 1, check=False) if s["nstep"]]
        err = sim.last_error()
        return stats, err, {n: sim.field(n) for n in FIELDS}, {n: sim.bubbles(n) for n in BUBBLES}


# one bubble a wavefront, a queue of lane pairs, a queue of lanes; the caps of the
# Picard iterations and of the RP sub-steps; a void fraction that leaves its range;
# little of it, so that every step ends with its first iteration, and then the sub-step cap or a
# state that overflows
@pytest.mark.parametrize("nb", [160, 2000, 9000])
@pytest.mark.parametrize("how", [{"max_picard": 1}, {"max_picard": 2}, {"max_picard": 4},
                                 {"max_substeps": 60}, {"max_substeps": 400},
                                 {"fg0": 0.05, "max_picard": 20, "max_substeps": 500},
                                 {"fg0": 1e-9, "max_substeps": 60},
                                 {"fg0": 1e-9, "max_substeps": 500, "poke": "PG"},
                                 {"fg0": 1e-9, "max_substeps": 500, "poke": "R_p"}])
@pytest.mark.parametrize("mixed", [0, 1])
def test_together_fails_as_one_at_a_time(brp, nb, how, mixed):
    how = dict(how)
    poke = how.pop("poke", None)
    cfg, b = cases.bubbly_case(64, nb=nb, seed=5, amp_pa=1.2e6, fg0=how.pop("fg0", 1e-5),
                               precision=brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64)
    cfg.update(**how)
    s1, e1, f1, b1 = run(brp, cfg, b, False, poke)
    s2, e2, f2, b2 = run(brp, cfg, b, True, poke)
    print(nb, how, poke, mixed, e1, "| iterations", "".join(str(s["n_pic"]) for s in s2), flush=True)
    assert e1 == e2 and s1 == s2
    for n in FIELDS:
        np.testing.assert_array_equal(f1[n], f2[n], err_msg=n)
    for n in BUBBLES:
        np.testing.assert_array_equal(b1[n], b2[n], err_msg=n)
