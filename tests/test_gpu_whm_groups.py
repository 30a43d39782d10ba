"""Whole WHM steps at the remainders of the pair groups of four, against the
oracle bit for bit."""
import numpy as np
import pytest

import pyoracle as O
import swiftest_amd as S
from swiftest_amd import ics

pytestmark = pytest.mark.gpu

KEYS = ("pl_rh", "pl_vh", "tp_rh", "tp_vh", "pl_status", "tp_status")


@pytest.mark.parametrize("lclose", [False, True])
@pytest.mark.parametrize("npl", [2, 3, 4, 5, 7, 9, 63])
def test_groups_of_four_bodies(npl, lclose):
    """The pair groups' remainders, with a mass outside the exact cores' range
    and, with radii, two bodies that overlap."""
    d = ics.whm_solar(seed=90 + npl, npl=npl, ntp=5)
    if lclose:
        d.Gmass[-1] = 1e-180
        if npl > 3:
            d.pl_rh[2] = d.pl_rh[1] * (1.0 + 1e-6)
            d.pl_vh[2] = d.pl_vh[1]
            d.radius[1] = d.radius[2] = 1e-4
    o = O.OracleSystem(O.WHM, d, 0.01, lclose=lclose)
    g = S.GpuSystem(S.WHM, d, 0.01, lclose=lclose)
    assert o.run(7) == 0
    g.run(7)
    a, b = o.state(), g.state()
    for k in KEYS:
        assert np.array_equal(a[k], b[k]), (npl, lclose, k)
