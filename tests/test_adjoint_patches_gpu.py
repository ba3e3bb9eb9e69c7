"""The motion transpose sums its node adjoints in LDS tiles, by the size of the
patch that a workgroup's 256 bubbles cover: vx and vy together, one after the
other, or each into the arrays.  The gradient of 256 bubbles against that of
the same bubbles among others of no weight (n_B = 0), which leave a workgroup
sixteen of them, on a patch that always fits."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


# cells a side: at most 2048 cells of the joint patch, at most 4096, more
@pytest.mark.parametrize("w,h", [(30, 40), (62, 44), (90, 60)])
@pytest.mark.parametrize("band", [1, 2, 3, 8])
def test_patch_forms_agree(brp, w, h, band):
    n, nb, steps = 110, 256, 150
    cfg, _ = cases.bubbly_case(n, nb=1, amp_pa=0.5e6, fg0=1e-8)
    cfg.sim_smooth_delta_band = band
    r = np.random.default_rng(10 * w + band)
    x, y = (12 + w * r.random(nb)) * 1e-4, (30 + h * r.random(nb)) * 1e-4
    R0 = 2e-6 + 2e-6 * r.random(nb)
    weight = 1e-8 * 1e-4**2 / (4 / 3 * np.pi * R0**3)  # a void fraction of 1e-8 in one cell
    source = (0.5e6 * (0.6 + 0.8 * r.random(4)), 0.3 * r.random(4))
    g = []
    for others in (0, 15):
        rep = 1 + others
        b = (np.repeat(x, rep), np.repeat(y, rep), np.repeat(R0, rep),
             np.repeat(weight, rep) * (np.arange(nb * rep) % rep == 0), 0.0)
        with cases.make(brp.Simulation, cfg, b, source) as sim:
            g.append(sim.adjoint((20, 90, 30, 80), steps, 60, 20))
    a, c = g
    assert a["J"] == c["J"] > 0.0
    # the same sums in another order of FP64 atomics
    for k in ("grad_amp", "grad_phase", "grad_fg0"):
        assert np.linalg.norm(c[k]) > 0.0
        assert np.linalg.norm(a[k] - c[k]) <= 1e-9 * np.linalg.norm(c[k]), k
