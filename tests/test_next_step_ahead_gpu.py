"""A step's first launches are queued before the host knows that the step
before ends: where that one goes on instead, they must leave everything as it
is.  Steps in one call (queued ahead) against one call a step (never), through
a collapse, in which the number of iterations changes."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


# one bubble a wavefront, a queue of lanes; the small and the large grid layout
@pytest.mark.parametrize("n,nb", [(64, 160), (64, 9000), (1100, 160)])
@pytest.mark.parametrize("mixed", [0, 1])
def test_together_equals_one_at_a_time(brp, n, nb, mixed):
    cfg, b = cases.bubbly_case(n, nb=nb, seed=5, amp_pa=1.2e6, fg0=1e-5,
                               precision=brp.abi.PREC_MIXED if mixed else brp.abi.PREC_FP64)
    one, many = cases.make(brp.Simulation, cfg, b), cases.make(brp.Simulation, cfg, b)
    steps = 130 if n == 64 else 40
    s1 = [one.step(1)[0] for _ in range(steps)]
    s2 = many.step(steps)
    pic = [s["n_pic"] for s in s2]
    print(n, nb, mixed, "iterations", "".join(map(str, pic)), flush=True)
    assert s1 == s2
    for f in ("R_t", "R_p", "PG", "Q_B", "sub", "PL_p", "x", "y", "vx", "vy"):
        np.testing.assert_array_equal(one.bubbles(f), many.bubbles(f), err_msg=f)
    for f in ("p0", "vx", "vy", "fg", "fgn"):
        np.testing.assert_array_equal(one.field(f), many.field(f), err_msg=f)
    if n == 64:
        assert any(a < c for a, c in zip(pic, pic[1:]))  # some went on past the guess
