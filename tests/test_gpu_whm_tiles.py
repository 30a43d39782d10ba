"""Whole WHM steps of systems with more particle tiles than the chip holds at
once (about 1024 tiles of 64): tiles that start after others have ended still
begin at the run's first state.  Against the per-step kernels, bit for bit."""
import numpy as np
import pytest

import swiftest_amd as S
from swiftest_amd import ics

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
