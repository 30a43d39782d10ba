"""Semi-interacting bodies (GMTINY) in systems that are loaded anew, against the
oracle's run of each alone, bit for bit: the first such bodies of an ensemble,
after steps that were captured without any, and slots with room to spare, whose
padding must not count among them."""
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


@pytest.mark.parametrize("cap,n,mlo", [(96, 60, 3e-4), (300, 33, 6e-4), (200, 90, 1e-5)])
@pytest.mark.parametrize("mode", [S.PAIR_EXACT, S.PAIR_FAST])
def test_padding_does_not_count_as_semi_interacting(cap, n, mlo, mode):
    """The accelerations themselves: a velocity hides the order of a sum."""
    print(f"gmtiny slot of {cap} with {n}, mode {mode}", flush=True)
    g = S.GpuSystem.slots(S.SYMBA, [cap], [10], 0.005, lclose=False, gmtiny=GT, pair_mode=mode)
    d = _disk(62 + n, n, mlo)
    tight = S.GpuSystem(S.SYMBA, d, 0.005, lclose=False, gmtiny=GT, pair_mode=mode)
    g.load(0, d)
    a, b = g.accel()[0][:n], tight.accel()[0]
    assert np.array_equal(a, b)
    if mode == S.PAIR_EXACT:
        k = np.argsort(-d.Gmass, kind="stable")
        nplm = int((d.Gmass >= GT).sum())
        assert 0 < nplm < n
        assert np.array_equal(a, O.accel_plpl(d.pl_rh[k], d.Gmass[k], d.radius[k], np.zeros((n, 3)), nplm=nplm))
