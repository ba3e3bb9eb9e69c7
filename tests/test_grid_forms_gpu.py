"""The grid kernels and their ghost cells against the oracle, from random
fields, in every combination of walls and sources, and on both sides of the
sizes where the split of a grid kernel changes.  Four steps of FP64 from the
same fields: each differs from the oracle by a few roundings a step (1e-12 of
the field's scale leaves a factor of a thousand)."""
import numpy as np
import pytest

import cases
import oracle_lib as ol

pytestmark = pytest.mark.gpu

FIELDS = ("p0", "px", "py", "vx", "vy")
SOURCES = ({}, {"tr_focused_p": 1}, {"tr_focused_v": 1}, {"tr_plane_v": 1},
           {"tr_plane_p": 1, "tr_plane_v": 1}, {"tr_focused_p": 1, "tr_focused_v": 1})


def config(brp, nx, ny, pml, source, bubbles=False, cyl=0):
    c = brp.abi.water_config(max(nx, ny), npml=2, bubbles=bubbles, focal_dist=0.6 * ny * 1e-4,
                             source_in_pml=False)
    c.update(grid_x=nx, grid_y=ny, grid_lx=nx * 1e-4, grid_ly=ny * 1e-4, tr_focused_p=0,
             ext_focus_x=0.4 * nx * 1e-4, tr_cylindrical=cyl,
             **{f"pml_{n}": pml >> k & 1 for k, n in enumerate(("x0", "x1", "y0", "y1"))})
    c.update(**source)
    return c


def check(brp, cfg, bubbles=None, steps=4, names=FIELDS):
    g = cases.make(brp.Simulation, cfg, bubbles)
    o = cases.make(ol.OracleSim, cfg, bubbles)
    r = np.random.default_rng(cfg.grid_x * 1000 + cfg.grid_y)
    for n in FIELDS:
        # beside bubbles small enough that the Picard loop converges
        a = r.standard_normal(g.shape(n)[1::-1]) * (1e5 if n[0] == "p" else 0.07)
        if bubbles is not None:
            a *= 1e-2
        g.set_field(n, a)
        o.set_field(n, a)
    gs, os_ = g.step(steps), o.step(steps)
    assert [s["n_pic"] for s in gs] == [s["n_pic"] for s in os_]
    for n in names:
        a, b = g.field(n), o.field(n)
        scale = max(np.abs(o.field(m)).max() for m in (FIELDS[:3] if n[0] == "p" else FIELDS[3:]))
        if n == "fg":
            scale = np.abs(b).max()
        assert np.abs(a - b).max() <= (1e-10 if n == "fg" else 1e-12) * scale, (n, cfg.grid_x, cfg.grid_y)
    g.close()
    o.close()


@pytest.mark.parametrize("pml", range(16))
def test_walls_and_sources(brp, pml):
    for nx, ny in ((7, 5), (5, 7), (6, 6), (9, 8), (8, 9), (10, 8)):
        for source in SOURCES:
            check(brp, config(brp, nx, ny, pml, source))
    check(brp, config(brp, 9, 11, pml, SOURCES[1], cyl=1))


# velocity splits at 2^20 cells, pressure at 300 000; ragged last columns and rows.
# x1 and y1 absorb: with a y1 mirror on a square grid the reference overwrites row M
# after each evaluation, so that its whole-grid residual never falls (kernel.cuh:929-932).
@pytest.mark.parametrize("nx,ny", [(1023, 1025), (1021, 1027), (1025, 1025), (257, 4097), (547, 548),
                                   (545, 551), (549, 547), (65, 4617)])
def test_both_splits(brp, nx, ny):
    r = np.random.default_rng(nx)
    n = 300
    x, y = nx * 1e-4 * r.random(n), ny * 1e-4 * r.random(n)
    cfg = config(brp, nx, ny, 0b1010, SOURCES[1], bubbles=True)
    check(brp, cfg, (x, y, np.full(n, 3e-6), None, 1e-6), steps=2, names=FIELDS + ("fg",))


@pytest.mark.parametrize("bubbles,thermal", [(0, 0), (1, 0), (1, 1), (0, 1)])
def test_phase_times_are_parts_of_the_call(brp, bubbles, thermal):
    import time
    cfg = config(brp, 200, 180, 15, SOURCES[1], bubbles=bool(bubbles))
    cfg.update(thermal=thermal)
    b = (np.full(1, 8e-3), np.full(1, 9e-3), np.full(1, 3e-6), None, 1e-6) if bubbles else None
    with cases.make(brp.Simulation, cfg, b) as sim:
        sim.step(5)
        t0 = time.perf_counter()
        n_pic = sum(s["n_pic"] for s in sim.step(40))
        wall = (time.perf_counter() - t0) * 1e3
        ph = sim.phase_times()
    assert all(v >= 0.0 for v in ph.values()) and ph["velocity"] > 0.0 and ph["pressure"] > 0.0
    assert (ph["motion"] > 0.0) == bool(bubbles) and (ph["bubble_rp"] > 0.0) == (n_pic > 0)
    assert ph["other"] > 0.0 or not thermal
    assert 0.2 * wall < sum(ph.values()) < wall, (ph, wall)
