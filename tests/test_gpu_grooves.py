"""Slip patterns through the fused path: the one-point front of odd theta
sizes with wall masks, and whole steps with oblique grooves at each row
capacity of the folded radial solve.  Tolerance: the 1e-10 relative L2 of the
workload contract."""
import pytest

from helpers import compare_fields, small_params, start_pair

pytestmark = pytest.mark.gpu

GROOVES = dict(minstrt=2, minstrz=3, multmin=1)


def _run(tc, oracle, p, steps, masks):
    dev, orc = start_pair(tc, oracle, p, 13, 1e-2)
    for n in range(steps):
        (c1, d1), (c2, d2) = dev.step(n), orc.step(n)
        assert c1 == c2 == 0 and d1["dt"] == d2["dt"]
    assert (dev.masks()[0].min() == 0) == masks
    compare_fields(dev, orc, p["nrm"], 1e-10)


@pytest.mark.parametrize("lpt", ["1", "2"])
@pytest.mark.parametrize("masks", [False, True])
def test_odd_theta_fronts_match_oracle(tc, oracle, monkeypatch, lpt, masks):
    """75 points: a full theta tile and a partial one; 54 z rows: a partial
    tile of four and of eight."""
    monkeypatch.setenv("TC_HELM_LPT", lpt)
    p = small_params(tc, 75, 54, 29, ntst=1000, sizepert=0.05, omegapert=0.3, virotext=0.2, romeg=0.1,
                     **(GROOVES if masks else {}))
    _run(tc, oracle, p, 4, masks)


@pytest.mark.parametrize("defer", ["0", "2"])
@pytest.mark.parametrize("nrm", [29, 100, 230, 300, 500, 801])
def test_grooved_steps_at_row_capacities(tc, oracle, monkeypatch, nrm, defer):
    monkeypatch.setenv("TC_DEFER_CORRECTION", defer)
    p = small_params(tc, 36, 24, nrm, ntst=1000, dtmin=1e-4, dtmax=1e-4, sizepert=0.1, omegapert=0.5,
                     **GROOVES)
    _run(tc, oracle, p, 3, True)


@pytest.mark.parametrize("nrm", [300, 500])
def test_grooved_odd_theta_steps(tc, oracle, nrm):
    p = small_params(tc, 45, 24, nrm, ntst=1000, dtmin=1e-4, dtmax=1e-4, **GROOVES)
    _run(tc, oracle, p, 3, True)
