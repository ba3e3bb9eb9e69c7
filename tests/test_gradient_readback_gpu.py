"""The gradient's map on a grid of more than 2^17 cells: the sum of three
arrays comes back in pieces, the first of which ends within a row, straight
into the caller's rows or row by row into longer ones."""
import ctypes as C

import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def test_map_in_pieces(brp):
    n, steps = 400, 40
    cfg, b = cases.bubbly_case(n, nb=30, amp_pa=0.5e6, fg0=1e-8)
    with cases.make(brp.Simulation, cfg, b, (np.full(4, 0.5e6), np.zeros(4))) as sim:
        nx, ny = sim.shape("fg")[:2]
        row, col = divmod(1 << 17, nx)  # where the first piece ends
        assert row < ny and 0 < col < nx
        box = (max(col - 15, 1), col + 15, row - 10, row + 10)
        r = np.random.default_rng(1)
        sim.set_field("p0", 1e3 * r.standard_normal(sim.shape("p0")[1::-1]))
        # a void fraction everywhere, so that every cell about the box has a derivative
        sim.set_field("fg", np.full((ny, nx), 1e-7))
        sim.save_state(0)
        g = sim.adjoint(box, steps, 10, 10)["grad_fg0"]
        sim.restore_state(0)
        out = np.full((ny, nx + 3), -7.0)
        ob = brp.abi.Objective(*box, steps, 10, 10, 0)
        sim._check(sim.lib.brp_adjoint(sim.h, C.byref(ob), None, None,
                                       out.ctypes.data_as(C.POINTER(C.c_double)), nx + 3, None))
    assert (g[row - 2:row + 3, box[0]:box[1] + 1] != 0.0).all()
    assert (out[:, nx:] == -7.0).all()
    # the same sums in another order of FP64 atomics
    assert np.abs(out[:, :nx] - g).max() <= 1e-9 * np.abs(g).max()
