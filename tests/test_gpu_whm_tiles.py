"""Whole WHM steps in one launch, against the per-step kernels bit for bit:
systems with more particle tiles than the chip holds at once (about 1024 tiles
of 64), whose late tiles still begin at the run's first state, and where a
failed drift stops the run."""
import numpy as np
import pytest

import swiftest_amd as S
from swiftest_amd import core, ics

pytestmark = pytest.mark.gpu

KEYS = ("pl_rh", "pl_vh", "tp_rh", "tp_vh", "pl_status", "tp_status", "lfirst")


@pytest.mark.parametrize("sizes", [((8, 150001),), ((3, 64), (5, 90000), (1, 0), (4, 65), (8, 70000))])
def test_more_tiles_than_fit(monkeypatch, sizes):
    print(f"whm tiles {sizes}", flush=True)
    systems = [ics.whm_solar(seed=40 + k, npl=n, ntp=t) for k, (n, t) in enumerate(sizes)]
    fused = S.GpuSystem(S.WHM, systems, 0.01)
    monkeypatch.setenv("SWG_WHM_STEPWISE", "1")
    stepwise = S.GpuSystem(S.WHM, systems, 0.01)
    monkeypatch.delenv("SWG_WHM_STEPWISE")
    for n in (3, 1, 2):  # a second and a third launch count from zero again
        fused.run(n)
        stepwise.run(n)
        a, b = fused.state(), stepwise.state()
        for k in KEYS:
            assert np.array_equal(a[k], b[k]), (n, k)


@pytest.mark.parametrize("step", [0, 1, 4, 11])
def test_failed_drift_stops_before_its_step(monkeypatch, step):
    """A body falling past the Sun at a speed its drift does not converge for:
    every particle, in all of the tiles, ends at the step before."""
    d = ics.whm_solar(seed=1, npl=3, ntp=700)
    speed = 24931.562736150383
    d.pl_rh[2] = speed * 0.01 * (step + 0.62) * np.array([0.6, 0.8, 0.0]) + 4e-8 * np.array([-0.8, 0.6, 0.0])
    d.pl_vh[2] = -speed * np.array([0.6, 0.8, 0.0])
    monkeypatch.setenv("SWG_WHM_STEPWISE", "1")
    probe, stepwise = (S.GpuSystem(S.WHM, d, 0.01, istep_out=0) for _ in range(2))
    monkeypatch.delenv("SWG_WHM_STEPWISE")
    good = 0
    with pytest.raises(core.SwiftestHipError):
        while good < 12:
            probe.step()
            good += 1
    assert good == step
    fused = S.GpuSystem(S.WHM, d, 0.01, istep_out=0)
    with pytest.raises(core.SwiftestHipError):
        fused.run(12)
    stepwise.run(good)
    a, b = fused.state(), stepwise.state()
    for k in ("tp_rh", "tp_vh", "tp_status"):
        assert np.array_equal(a[k], b[k]), (step, k)
    assert np.count_nonzero(a["pl_status"]) == 1
