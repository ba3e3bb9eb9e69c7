"""The smooth-delta stencils: the band known at compile time (2) and the
general one (the others) against the oracle: motion, gather and scatter."""
import pytest

import cases
from oracle_lib import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("band", [1, 2, 3, 4, 8])
def test_bands_match_the_oracle(brp, band):
    cfg, b = cases.bubbly_case(48, nb=90, seed=band, amp_pa=4.0e5)
    cfg.sim_smooth_delta_band = band
    g = cases.make(brp.Simulation, cfg, b)
    o = cases.make(OracleSim, cfg, b)
    g.step(60)
    o.step(60)
    # positions, velocities and radii: one forward's accumulated rounding, as
    # the other oracle comparisons of unbroken fp64 runs
    for n in ("x", "y", "vx", "vy", "R_t", "PL_p"):
        assert cases.rel_l2(g.bubbles(n), o.bubbles(n)) < 1e-9, n
    for f in ("p0", "fg"):
        assert cases.rel_l2(g.field(f), o.field(f)) < 1e-9, f
