"""Steps of acoustics alone are queued ahead of the host's reading of their
reports: the same fields and stats as one at a time, and after a step that
fails the same state, as if the steps behind it had not been queued."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

FIELDS = ("p0", "px", "py", "vx", "vy")


# below and above the grid sizes at which the velocity and pressure kernels
# change their layout; fewer, as many and more steps than are queued ahead
@pytest.mark.parametrize("n", [48, 640, 1100])
@pytest.mark.parametrize("steps", [3, 8, 29])
def test_together_equals_one_at_a_time(brp, n, steps):
    cfg = brp.abi.water_config(n, npml=8)
    a, b = cases.make(brp.Simulation, cfg), cases.make(brp.Simulation, cfg)
    sa = a.step(steps)
    sb = [b.step(1)[0] for _ in range(steps)]
    assert sa == sb
    for f in FIELDS:
        np.testing.assert_array_equal(a.field(f), b.field(f))
    assert a.step(2) == b.step(1) + b.step(1)


@pytest.mark.parametrize("n", [48, 1100])
def test_a_failed_step_stops_the_ones_behind_it(brp, n):
    cfg = brp.abi.water_config(n, npml=8, precision=brp.abi.PREC_MIXED, amp_pa=3.0e38)
    a, b = cases.make(brp.Simulation, cfg), cases.make(brp.Simulation, cfg)
    for s in (a, b):
        s.save_state(0)
    with pytest.raises(Exception) as ea:
        a.step(60)
    n_ok = 0
    with pytest.raises(Exception) as eb:
        for _ in range(60):
            b.step(1)
            n_ok += 1
    assert 1 <= n_ok < 59, n_ok  # some pass first, and more than those ahead follow
    assert str(ea.value) == str(eb.value)
    for f in FIELDS:
        np.testing.assert_array_equal(a.field(f), b.field(f))
    for s in (a, b):
        s.restore_state(0)
    assert a.step(n_ok) == [b.step(1)[0] for _ in range(n_ok)]
