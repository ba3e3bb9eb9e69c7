"""An RP call that a step did not need (test_rp_ahead_gpu) with the
operation-by-operation sub-step, which always takes the queue of lanes, and
with the fold at the axis."""
import pytest

import test_rp_ahead_gpu as ahead

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [300, 2000, 9000])
@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("option", ["rp_exact", "tr_cylindrical"])
def test_unneeded_call_changes_nothing(brp, nb, mixed, option, monkeypatch):
    bubbly = ahead.cases.bubbly_case

    def with_option(*a, **k):
        cfg, b = bubbly(*a, **k)
        return cfg.update(**{option: 1}), b

    monkeypatch.setattr(ahead.cases, "bubbly_case", with_option)
    ahead.test_unneeded_call_changes_nothing(brp, nb, mixed)
