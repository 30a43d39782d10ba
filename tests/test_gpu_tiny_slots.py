"""Semi-interacting bodies (GMTINY) in systems that are loaded anew, against the
oracle's run of each alone, bit for bit: the first such bodies of an ensemble,
after steps that were captured without any."""
import numpy as np
import pytest

import pyoracle as O
import swiftest_amd as S
from helpers import compact_disk
from swiftest_amd import ics

pytestmark = pytest.mark.gpu

GT = 1e-3 * ics.GU
KEYS = ("pl_rh", "pl_vh", "pl_vb", "tp_rh", "tp_vh", "tp_vb", "pl_status", "tp_status")


def _disk(seed, n, mlo):
    return compact_disk(seed=seed, npl=n, ntp=10, mlo=mlo, mhi=1e-2, alo=0.5, ahi=30.0)


def _run_slot(g, sysic, label, steps=3):
    o = O.OracleSystem(O.SYMBA, sysic, 0.005, gmtiny=GT, lclose=False)
    g.load(0, sysic)
    for k in range(steps):
        assert o.run(1) == 0
        g.run(1)
        a, b = o.state(), g.get_slot(0)
        for key in KEYS:
            assert np.array_equal(a[key], b[key]), (label, k, key)


def test_first_semi_interacting_bodies_after_captured_steps():
    n = 80
    heavy = _disk(60, n, 2e-3)
    mixed = _disk(61, n, 3e-4)
    assert (heavy.Gmass >= GT).all() and 0 < (mixed.Gmass < GT).sum() <= n // 2
    g = S.GpuSystem(S.SYMBA, heavy, 0.005, lclose=False, gmtiny=GT)
    g.use_graphs(True)
    _run_slot(g, heavy, "heavy")
    _run_slot(g, mixed, "mixed")
