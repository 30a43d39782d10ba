"""GPU parity of the recursion's one-wavefront mode at its edges: up to 64
bodies, pairs and kick entries, one to the limit and one past it, bound
bodies (drifted on the first wavefront), unbound ones (on the others, two
lanes a body sharing its two cube roots) and particles among them."""
import numpy as np
import pytest

import pyoracle as O
import swiftest_amd as S
from swiftest_amd import ics

pytestmark = pytest.mark.gpu


def tight_pairs(npairs, unbound, ntp, seed=3):
    """npairs close pairs of bodies around the star, far from one another,
    the first `unbound` of them on hyperbolic orbits, and ntp particles each
    beside one body."""
    rng = np.random.Generator(np.random.PCG64(seed))
    phi = 2 * np.pi * np.arange(npairs) / max(npairs, 1)
    c = np.stack([np.cos(phi), np.sin(phi), 0 * phi], 1)
    t = np.stack([-np.sin(phi), np.cos(phi), 0 * phi], 1)
    r = np.repeat(c, 2, axis=0)
    v = np.where((np.arange(npairs) < unbound)[:, None], 10.0 * c, 2 * np.pi * t).repeat(2, axis=0)
    gap = rng.uniform(1e-4, 3e-4, npairs)
    r[0::2] += gap[:, None] * t
    r[1::2] -= gap[:, None] * t
    v[0::2, 2] += 0.02
    m = rng.uniform(1e-8, 2e-8, 2 * npairs)
    Gm = ics.GU * m
    R = 0.01 * ics._radius_from_mass(m)
    q = rng.integers(0, 2 * npairs, ntp)
    tr, tv = r[q] + rng.normal(0, 2e-4, (ntp, 3)), v[q] + rng.normal(0, 1e-2, (ntp, 3))
    return ics.System(ics.GMSUN, ics.RSUN_AU, r, v, Gm, R, tr, tv)


@pytest.mark.parametrize("npairs,unbound,ntp,sc", [(1, 0, 0, True), (1, 1, 0, True), (31, 31, 0, True),
                                                   (32, 17, 0, True), (32, 32, 0, True), (33, 20, 0, True),
                                                   (12, 6, 20, False), (12, 6, 20, True), (2, 1, 64, False)])
def test_wave_mode_edges(npairs, unbound, ntp, sc):
    print(f"wave mode npairs={npairs} unbound={unbound} ntp={ntp} short_circuit={sc}", flush=True)
    sysic = tight_pairs(npairs, unbound, ntp)
    o = O.OracleSystem(O.SYMBA, sysic, 0.002, short_circuit=sc, lclose=False)
    g = S.GpuSystem(S.SYMBA, sysic, 0.002, short_circuit=sc, lclose=False)
    for step in range(3):
        assert o.run(1) == 0
        g.run(1)
        so, sg = o.stats(), g.stats()
        assert (so["max_depth"], so["nsubsteps"], so["npltp_enc"]) == (sg["max_depth"], sg["nsubsteps"],
                                                                       sg["npltp_enc"]), (step, so, sg)
        a, b = o.state(), g.state()
        assert np.array_equal(a["tp_status"], b["tp_status"]) and np.array_equal(a["pl_status"], b["pl_status"])
        for k in ("pl_rh", "pl_vh", "tp_rh", "tp_vh"):
            if unbound == 0:
                assert np.array_equal(a[k], b[k]), (step, k)
            elif a[k].size:
                # the starting guess of an unbound drift is a cube root, where
                # the host library's pow differs from the correctly rounded one
                # by an ulp in 0.08 % of its calls: about 40 of a step's 2.6e4
                # drifts, 2^-52 of the state each, magnified up to a few
                # hundred times by three steps of the pairs' own motion
                # (40 * 2.2e-16 * 1e3 = 9e-12)
                d = np.abs(a[k] - b[k]).max() / np.abs(a[k]).max()
                assert d <= 1e-11, (step, k, d)
    assert sg["max_depth"] >= 4
