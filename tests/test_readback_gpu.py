"""Read-back of fields and bubble arrays: pieces of 2^17 values through pinned
slots, rows cut at piece edges, against the values set."""
import ctypes as C

import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def get(sim, brp, name, ld):
    fid = brp.abi.FIELD_NAMES[name]
    nx, ny, _, _ = sim.shape(fid)
    out = np.full((ny, ld or nx), -7.0)
    sim._check(sim.lib.brp_get_field(sim.h, fid, out.ctypes.data_as(C.POINTER(C.c_double)), ld or nx))
    return out[:, :nx], out[:, nx:]


# one slot; a value less and more than one slot's 2^17 (361 * 363 = 131043,
# 364 * 362 = 131768); a few pieces; pieces for every thread, the last one ragged
@pytest.mark.parametrize("nx,ny", [(5, 4), (359, 361), (362, 360), (700, 513), (1500, 1201)])
@pytest.mark.parametrize("mixed", [0, 1])
def test_fields_come_back_as_set(brp, nx, ny, mixed):
    cfg = brp.abi.water_config(max(nx, ny), npml=2, bubbles=False,
                               precision=brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64)
    cfg.update(grid_x=nx, grid_y=ny, grid_lx=nx * 1e-4, grid_ly=ny * 1e-4)
    r = np.random.default_rng(nx)
    with brp.Simulation(cfg) as sim:
        sim.prepare()
        for name in ("p0", "vx", "vy", "fg"):
            a = r.standard_normal(sim.shape(name)[1::-1]).astype(np.float32).astype(np.float64)
            if name == "fg":
                a = np.rint(a * 2.0**50) * 2.0**-55  # whole numbers of 2^-60 below 1
                a = np.clip(a, -0.5, 0.5)
            sim.set_field(name, a)
            np.testing.assert_array_equal(sim.field(name), a)
            for ld in (a.shape[1] + 3,):
                got, rest = get(sim, brp, name, ld)
                np.testing.assert_array_equal(got, a)
                assert (rest == -7.0).all()
        np.testing.assert_array_equal(sim.field("fgn"), sim.field("fg"))


@pytest.mark.parametrize("nb", [1, 1000, (1 << 17) + 1, 700001])
def test_bubbles_come_back_in_the_callers_order(brp, nb):
    cfg, _ = cases.bubbly_case(64, nb=1)
    r = np.random.default_rng(nb)
    x, y = (r.random(nb) * 6e-3 for _ in range(2))
    R0 = 1e-6 + 4e-6 * r.random(nb)
    with brp.Simulation(cfg) as sim:
        sim.set_bubbles(x, y, R0, None, 1e-9)
        sim.prepare()
        for name, a in (("x", x), ("y", y), ("R0", R0), ("R_t", R0), ("sub", np.zeros(nb))):
            np.testing.assert_array_equal(sim.bubbles(name), a)
        info = sim.info()
        np.testing.assert_array_equal(sim.bubbles("ibn_x"), np.floor(x * info["rdx"] + 0.5))
