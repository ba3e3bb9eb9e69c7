"""Gradients on a grid of more rows than a step record's copies take workgroups
in y: two bubbles without weight at the far ends stretch the Picard window over
all rows, and no derivative near the middle changes with them."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [0, 1])
def test_far_rows_are_recorded(brp, mixed):
    nx, ny, h, steps = 12, 40000, 1e-4, 12
    cfg = brp.abi.water_config(nx, npml=2, focal_dist=0.6 * ny * h,
                               precision=brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64)
    cfg.update(grid_x=nx, grid_y=ny, grid_lx=nx * h, grid_ly=ny * h)
    r = np.random.default_rng(1)
    nb, mid = 30, 36000
    x, y = (4 + 4 * r.random(nb)) * h, (mid + 6 * r.random(nb)) * h
    R0 = 2e-6 + 2e-6 * r.random(nb)
    weight = 1e-7 * h**2 / (4 / 3 * np.pi * R0**3)
    p = np.zeros((ny + 2, nx + 2))
    p[mid - 20:mid + 30] = 1e4 * r.standard_normal((50, nx + 2))
    g = []
    for ends in (0, 2):
        b = (np.append(x, [6 * h] * ends), np.append(y, [6 * h, (ny - 6) * h][:ends]),
             np.append(R0, [3e-6] * ends), np.append(weight, [0.0] * ends), 0.0)
        with cases.make(brp.Simulation, cfg, b, (np.full(2, 1e5), np.zeros(2))) as sim:
            assert sim.shape("p0")[1::-1] == p.shape
            sim.set_field("p0", p)
            g.append(sim.adjoint((2, 11, mid - 4, mid + 10), steps, 4, 6))
            assert sim.bubbles("sub")[:nb].min() > 0
    a, c = g
    assert a["J"] == c["J"] > 0.0
    # cells of both windows
    u, v = (q["grad_fg0"][mid + 1:mid + 6, 5:8] for q in g)
    assert (u != 0.0).all()
    # the same sums in another order of FP64 atomics
    assert np.abs(u - v).max() <= 1e-9 * np.abs(u).max()
