"""GPU parity of the row kernels (terms evaluated by several wavefronts, folded
in partner order) at the edges of their 16- and 64-body tiles and 64-partner
chunks, against the oracle bit for bit."""
import numpy as np
import pytest

import pyoracle as O
import swiftest_amd as S
from helpers import compact_disk
from swiftest_amd import ics

pytestmark = pytest.mark.gpu


def _bodies(n, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    r = rng.normal(0, 2.0, (n, 3))
    Gm = ics.GU * np.exp(rng.uniform(np.log(1e-9), np.log(1e-3), n))
    R = np.exp(rng.uniform(np.log(1e-5), np.log(1e-2), n))
    return rng, r, Gm, R


@pytest.mark.parametrize("n,nplm", [(1, 1), (1, 0), (2, 1), (15, 15), (16, 16), (17, 9), (63, 32), (64, 64), (65, 31),
                                    (65, 33), (79, 79), (129, 64), (129, 65), (200, 0), (333, 17), (1000, 1000)])
@pytest.mark.parametrize("with_radius", [True, False])
def test_rows_at_tile_edges(n, nplm, with_radius):
    print(f"rows n={n} nplm={nplm} radius={with_radius}", flush=True)
    rng, r, Gm, R = _bodies(n, 7 * n + nplm)
    if n > 20:
        r[18] = r[3] + 1e-3  # overlapping: left out when radii are used
        Gm[5] = 0.0
    acc = rng.normal(0, 1e-3, (n, 3))
    acc[0] = -0.0            # a sum that starts at -0 and may get no term
    rad = R if with_radius else None
    ref = O.accel_plpl(r, Gm, rad, acc, nplm=nplm)
    got = S.swiftest_kick_getacch_int_all_tri(n, nplm, r, Gm, rad, acc)
    assert np.array_equal(ref.view(np.int64), got.view(np.int64))


@pytest.mark.parametrize("n,nplm", [(4096, 4096), (4097, 2100), (10007, 10007), (12287, 6200), (12288, 12288), (12351, 6200),
                                    (6001, 2000)])
@pytest.mark.parametrize("with_radius", [True, False])
def test_large_systems_at_tile_edges(n, nplm, with_radius):
    """Either side of the limits between the row kernels (4096 bodies, 192
    tiles of 64), partial last tiles and a first semi-interacting body inside a
    tile; overlapping bodies, two at one place, a body at NaN (left out with
    radii) and masses outside the exact cores' range in some chunks."""
    print(f"large rows n={n} nplm={nplm} radius={with_radius}", flush=True)
    rng, r, Gm, R = _bodies(n, n + nplm)
    r[n // 2] = r[n // 2 + 1] + 1e-3
    R[n // 2] = R[n // 2 + 1] = 1e-2
    r[700] = r[900]
    Gm[1500], Gm[n - 1], Gm[64] = 1e-200, 1e-170, 0.0
    acc = rng.normal(0, 1e-3, (n, 3))
    acc[0] = acc[n - 1] = -0.0
    rad = R if with_radius else None
    ref = O.accel_plpl(r, Gm, rad, acc, nplm=nplm)
    got = S.swiftest_kick_getacch_int_all_tri(n, nplm, r, Gm, rad, acc)
    assert np.array_equal(ref, got, equal_nan=True)
    if with_radius:
        assert np.isfinite(ref).all()
        assert np.array_equal(ref.view(np.int64), got.view(np.int64))
        r[2100, 1] = np.nan
        ref = O.accel_plpl(r, Gm, rad, acc, nplm=nplm)
        got = S.swiftest_kick_getacch_int_all_tri(n, nplm, r, Gm, rad, acc)
        assert np.isfinite(ref).all()
        assert np.array_equal(ref.view(np.int64), got.view(np.int64))


@pytest.mark.parametrize("n,nplm", [(70, 70), (70, 20)])
def test_rows_outside_the_fast_range(n, nplm):
    """Separations and masses outside the exact cores' range, then a body at
    NaN, which radii leave out of every other's sum, and one at infinity, which
    they do not, bit for bit."""
    rng, r, Gm, R = _bodies(n, 5)
    r[:10] *= 1e-130
    r[10:20] *= 1e130
    Gm[30] = 1e-200
    acc = np.zeros((n, 3))
    ref = O.accel_plpl(r, Gm, None, acc, nplm=nplm)
    got = S.swiftest_kick_getacch_int_all_tri(n, nplm, r, Gm, None, acc)
    assert np.array_equal(ref, got, equal_nan=True)
    r[40] = np.nan
    ref = O.accel_plpl(r, Gm, R, acc, nplm=nplm)
    got = S.swiftest_kick_getacch_int_all_tri(n, nplm, r, Gm, R, acc)
    assert np.isfinite(np.delete(ref, slice(0, 20), 0)).all()
    assert np.array_equal(ref, got, equal_nan=True)
    r[50] = np.inf
    ref = O.accel_plpl(r, Gm, R, acc, nplm=nplm)
    got = S.swiftest_kick_getacch_int_all_tri(n, nplm, r, Gm, R, acc)
    assert np.array_equal(ref, got, equal_nan=True)


@pytest.mark.parametrize("q,pm", [(0.0, "exact"), (0.3, "exact"), (0.7, "exact"), (0.7, "fast")])
@pytest.mark.parametrize("n", [33, 130])
def test_rows_with_encounter_pairs(n, q, pm):
    """Resident kicks with encounter-pair removal, with and without
    semi-interacting bodies (both branches): 4 steps of a crowded disk."""
    d = compact_disk(seed=50 + n, npl=n, ntp=10, mlo=1e-8, mhi=1e-5)
    gmt = float(np.quantile(d.Gmass, q)) if q else 0.0
    fast = pm == "fast"
    o = O.OracleSystem(O.SYMBA, d, 0.005, gmtiny=gmt, lclose=False)
    g = S.GpuSystem(S.SYMBA, d, 0.005, gmtiny=gmt, lclose=False, pair_mode=S.PAIR_FAST if fast else S.PAIR_EXACT)
    for k in range(4):
        assert o.run(1) == 0
        g.run(1)
        a, b = o.state(), g.state()
        for key in ("pl_rh", "pl_vb", "tp_rh", "tp_vb"):
            if fast:
                # a few ulp per factor, magnified by the encounters
                assert np.abs(a[key] - b[key]).max() <= 1e-10 * np.abs(a[key]).max(), (k, key)
            else:
                assert np.array_equal(a[key], b[key]), (k, key)
    assert g.stats()["nplpl_enc"] > 0


@pytest.mark.parametrize("npl,ntp", [(1, 1), (3, 65), (4, 63), (31, 16), (32, 1), (32, 16), (33, 17), (63, 15), (64, 64),
                                     (65, 100), (129, 33), (500, 1000), (67, 40960), (67, 40961)])
def test_particles_at_tile_edges(npl, ntp):
    """Particle sums by rows and by lanes (few massive bodies, many particles),
    with masked particles, massless bodies and some separations and masses
    outside the exact cores' range."""
    print(f"particles npl={npl} ntp={ntp}", flush=True)
    rng, r, Gm, _ = _bodies(npl, npl + ntp)
    rt = rng.normal(0, 2.0, (ntp, 3))
    mask = (rng.random(ntp) > 0.1).astype(np.int32)
    acc = rng.normal(0, 1e-3, (ntp, 3))
    acc[0] = -0.0
    ref = O.accel_pltp(rt, r, Gm, mask, acc)
    got = S.swiftest_kick_getacch_int_all_tp(ntp, npl, rt, r, Gm, mask, acc)
    assert np.array_equal(ref.view(np.int64), got.view(np.int64))
    Gm[npl // 2] = 0.0
    Gm[-1] = 1e-200
    rt[ntp // 2] *= 1e130
    rt[-1] = r[0] + 1e-130
    ref = O.accel_pltp(rt, r, Gm, mask, acc)
    got = S.swiftest_kick_getacch_int_all_tp(ntp, npl, rt, r, Gm, mask, acc)
    assert np.array_equal(ref, got, equal_nan=True)
    if ntp > 1000:
        return
    S.set_pair_mode(S.PAIR_FAST)
    try:
        fast = S.swiftest_kick_getacch_int_all_tp(ntp, npl, rt, r, Gm, mask, np.zeros((ntp, 3)))
    finally:
        S.set_pair_mode(S.PAIR_EXACT)
    ref = O.accel_pltp(rt, r, Gm, mask, np.zeros((ntp, 3)))
    keep = np.arange(ntp)
    keep = keep[(keep != ntp // 2) & (keep != ntp - 1)]  # the others' factors leave the normal range
    d = rt[keep, None, :] - r[None, :, :]
    terms = (Gm[None, :, None] * np.abs(d) / ((d * d).sum(-1) ** 1.5)[..., None]).sum(1)
    # each factor within 8 ulp of the exact mode's, then npl roundings of partial
    # sums no larger than the sum of the terms' sizes, on both sides
    assert (np.abs(fast - ref)[keep] <= 2 * (npl + 8) * 2.0**-52 * terms).all()


def test_ensemble_of_short_systems():
    """An ensemble large enough for the kernel with one body per lane, its
    systems at the edges of the 64-body tiles and 64-partner chunks, one of
    them with overlapping bodies and masses outside the exact cores' range."""
    sizes = [17, 63, 64, 65, 100, 127, 128, 129, 1] * 36
    systems = [compact_disk(seed=200 + k % 18, npl=n, mlo=1e-8, mhi=1e-3) for k, n in enumerate(sizes)]
    d = systems[7]
    d.pl_rh[40] = d.pl_rh[90] + 1e-7
    d.radius[40] = d.radius[90] = 1e-5
    d.Gmass[3], d.Gmass[100] = 1e-180, 0.0
    g = S.GpuSystem(S.SYMBA, systems, 0.005, lclose=False)
    st, (a, _) = g.state(), g.accel()
    off = np.cumsum([0] + sizes)
    for k in range(18):
        s, ids = slice(off[k], off[k + 1]), st["pl_id"][off[k]:off[k + 1]] - 1
        ref = O.accel_plpl(st["pl_rh"][s], systems[k].Gmass[ids], systems[k].radius[ids])
        assert np.array_equal(ref, a[s]), k
    for k in range(18, len(sizes)):
        if k % 18 != 7:
            assert np.array_equal(a[off[k]:off[k + 1]], a[off[k % 18]:off[k % 18 + 1]]), k
