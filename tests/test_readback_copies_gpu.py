"""Read-back of the arrays that are copied as they are and converted on the host
(16 to 64 KiB), of those below and above: every kind of value."""
import numpy as np
import pytest

import cases
from test_readback_gpu import get
from test_zz_no_alloc import _both

pytestmark = pytest.mark.gpu


# frames of 64-element rows: FP64 and the void fraction are copied from 15 x 13 to 50 x 37 and at
# 300 x 8, FP32 from 60 x 40 to 110 x 60; at 64 x 40 rows are 192 long
@pytest.mark.parametrize("nx,ny", [(5, 4), (15, 13), (50, 37), (50, 60), (60, 40), (64, 40), (110, 60),
                                   (110, 80), (300, 8), (300, 20)])
@pytest.mark.parametrize("mixed", [0, 1])
def test_fields(brp, nx, ny, mixed):
    cfg = brp.abi.water_config(max(nx, ny), npml=2, bubbles=False,
                               precision=brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64)
    cfg.update(grid_x=nx, grid_y=ny, grid_lx=nx * 1e-4, grid_ly=ny * 1e-4, thermal=1)
    r = np.random.default_rng(nx * ny)
    with brp.Simulation(cfg) as sim:
        sim.prepare()
        sim.step(1)  # the density is the void fraction's from the second step on
        for name in ("p0", "px", "py", "vx", "vy", "fg", "T"):
            a = r.standard_normal(sim.shape(name)[1::-1]).astype(np.float32).astype(np.float64)
            if name == "fg":
                a = np.clip(np.rint(a * 2.0**50) * 2.0**-55, -0.5, 0.5)
            sim.set_field(name, a)
            for pad in (0, 3):
                got, rest = get(sim, brp, name, a.shape[1] + pad)
                np.testing.assert_array_equal(got, a, err_msg=name)
                assert (rest == -7.0).all()
            if name == "fg":
                np.testing.assert_array_equal(sim.field("rho_m"), (1.0 - a) * 1000.0)


@pytest.mark.parametrize("nb", [2047, 2048, 4095, 4096, 8192, 8193, 16384, 16385])
def test_bubbles(brp, nb):
    cfg, b = cases.bubbly_case(48, nb=nb, seed=nb, amp_pa=1.5e6)
    with cases.make(brp.Simulation, cfg, b) as sim:
        sim.step(90)  # collapsing
        assert len(np.unique(sim.bubbles("sub"))) > 1
        for name in brp.abi.BUB_NAMES:
            a, c = _both(brp, sim, name)
            np.testing.assert_array_equal(a, c, err_msg=name)
