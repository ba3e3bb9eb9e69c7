"""The gradient by a recomputation that integrates RP (no tape) against one
that replays the tape without waiting, for stencil bands of both kernel forms
and a population whose patches do not fit the LDS tiles."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def gradient(brp, cfg, b, source, steps, tape, every=7):
    with cases.make(brp.Simulation, cfg, b, source) as sim:
        return sim.adjoint(cases.focal_box(cfg), steps, 6, every, tape=tape), sim.field("p0")


# bands: one cell, the reference's, an odd one, the largest; bubbles: few over a
# wide box (patches larger than a tile), and a prime number over several workgroups
@pytest.mark.parametrize("band", [1, 2, 3, 8])
@pytest.mark.parametrize("nb,box,n", [(37, 9.5e-3, 110), (521, 2e-3, 56)])
def test_tape_and_recomputation_agree(brp, band, nb, box, n):
    cfg, b = cases.bubbly_case(n, nb=nb, seed=nb + band, amp_pa=0.8e6, box=box, fg0=1e-8)
    cfg.sim_smooth_delta_band = band
    r = np.random.default_rng(band)
    source = (0.8e6 * (0.6 + 0.8 * r.random(4)), 0.3 * r.random(4))
    (a, pa), (c, pc) = (gradient(brp, cfg, b, source, 2 * n, tape) for tape in (True, False))
    np.testing.assert_array_equal(pa, pc)
    assert a["J"] == c["J"] and a["schedule_mismatch"] == c["schedule_mismatch"] == 0
    # the same sums in another order of FP64 atomics
    for k in ("grad_amp", "grad_phase", "grad_fg0"):
        assert np.linalg.norm(a[k] - c[k]) <= 1e-9 * np.linalg.norm(c[k]), k
