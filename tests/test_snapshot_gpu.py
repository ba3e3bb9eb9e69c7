"""Snapshots hold the void fraction on the rows of the Picard window only: a
restore must also clear the rows that the window has reached since, and a slot
saved again must hold a window that has grown."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

FIELDS = ("p0", "px", "py", "vx", "vy", "fg", "fgn", "fgm")
BUBBLES = ("x", "y", "R_t", "R_p", "R_n", "d1R", "PG", "PL_p", "PL_n", "PL_m", "Q_B", "dt", "re", "sub")


def state(sim):
    s = {n: sim.field(n) for n in FIELDS}
    if sim.info()["n_bubbles"]:
        s.update({"b_" + n: sim.bubbles(n) for n in BUBBLES})
    return s


def same(a, b):
    for n in a:
        np.testing.assert_array_equal(a[n], b[n], err_msg=n)


# bubbles: none, one, an odd number (arrays of 4 bytes a bubble end in a part of a 16-byte piece)
@pytest.mark.parametrize("nb", [0, 1, 33, 1027])
@pytest.mark.parametrize("mixed", [0, 1])
def test_restore_after_the_window_has_grown(brp, nb, mixed):
    prec = brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64
    cfg, b = cases.bubbly_case(64, nb=max(nb, 1), seed=nb, precision=prec)
    cfg.bub_enable = int(nb > 0)
    with cases.make(brp.Simulation, cfg, b if nb else None) as sim:
        sim.step(40)
        sim.save_state(0)
        s0 = state(sim)
        sim.step(7)
        s7 = state(sim)
        sim.restore_state(0)
        same(state(sim), s0)
        far = np.zeros(sim.shape("fgn")[1::-1])
        far[3, 5] = far[60, 2] = 2.0**-20  # rows below and above the saved window
        sim.set_field("fgn", far)
        sim.save_state(3)
        sim.save_state(0)  # the slot's block grows
        big = state(sim)
        sim.step(3)
        sim.restore_state(0)
        same(state(sim), big)
        sim.set_field("fgn", s0["fgn"])
        sim.save_state(1)
        sim.restore_state(3)
        same(state(sim), big)
        sim.restore_state(1)
        same(state(sim), s0)
        sim.step(7)
        same(state(sim), s7)
