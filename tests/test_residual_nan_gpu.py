"""The first evaluation's residual is that of the cells that hold a number:
one workgroup's cells of the one-cell-per-thread form are all set to NaN."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def run(brp, nx, ny, mixed, nan, bubbles):
    cfg = brp.abi.water_config(max(nx, ny), npml=2, bubbles=bubbles, focal_dist=0.6 * ny * 1e-4,
                               precision=brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64)
    cfg.update(grid_x=nx, grid_y=ny, grid_lx=nx * 1e-4, grid_ly=ny * 1e-4,
               ext_focus_x=0.4 * nx * 1e-4)
    n = 20
    r = np.random.default_rng(nx)
    b = (160e-4 + 10e-4 * r.random(n), 28e-4 + 4e-4 * r.random(n), np.full(n, 3e-6), None, 1e-8)
    with cases.make(brp.Simulation, cfg, b if bubbles else None) as sim:
        a = (1e3 * r.standard_normal(sim.shape("p0")[1::-1])).astype(np.float32).astype(np.float64)
        if nan:
            a[8:12, 64:128] = np.nan  # rows 8..11, columns 64..127 of 64 x 4 threads
        sim.set_field("p0", a)
        return a, sim.step(1, check=False)[0], sim.field("p0")


# both forms of the pressure evaluation (300 000 cells)
@pytest.mark.parametrize("nx,ny", [(200, 40), (700, 600)])
@pytest.mark.parametrize("mixed", [0, 1])
def test_the_residual_passes_over_nan(brp, nx, ny, mixed):
    a, s, p = run(brp, nx, ny, mixed, True, False)
    assert s["status"] == brp.abi.ERR_NONFINITE
    # the same difference of doubles, over the ambient pressure
    assert s["resimax0"] == np.nanmax(np.abs(a - p)[1:-1, 1:-1]) / 0.1e6


@pytest.mark.parametrize("nx,ny", [(200, 40), (700, 600)])
@pytest.mark.parametrize("mixed", [0, 1])
def test_picard_runs_beside_nan(brp, nx, ny, mixed):
    clean = run(brp, nx, ny, mixed, False, True)[1]
    s = run(brp, nx, ny, mixed, True, True)[1]
    assert s["status"] == brp.abi.ERR_NONFINITE and clean["status"] == 0
    assert s["n_pic"] == clean["n_pic"] > 0 and s["resimax"] == clean["resimax"]
