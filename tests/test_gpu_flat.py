"""Pair-list sums: lists in any order, at the edges of the fold's groups of
sixteen and of a round of pairs, against the oracle bit for bit."""
import numpy as np
import pytest

import pyoracle as O
import swiftest_amd as S
from swiftest_amd import core, ics

pytestmark = pytest.mark.gpu


def _bodies(n, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    r = rng.normal(0, 2.0, (n, 3))
    Gm = ics.GU * np.exp(rng.uniform(np.log(1e-9), np.log(1e-3), n))
    R = np.exp(rng.uniform(np.log(1e-5), np.log(1e-2), n))
    acc = rng.normal(0, 1e-3, (n, 3))
    acc[0] = -0.0
    return rng, r, Gm, R, acc


@pytest.mark.parametrize("n,m", [(1, 0), (1, 3), (2, 1), (2, 16), (2, 17), (3, 31), (15, 33), (16, 200), (17, 64), (300, 0),
                                 (300, 3000), (129, 40000), (1000, (1 << 20) + 3)])
@pytest.mark.parametrize("with_radius", [True, False])
def test_lists_in_any_order(n, m, with_radius):
    print(f"flat n={n} m={m} radius={with_radius}", flush=True)
    rng, r, Gm, R, acc = _bodies(n, n + m)
    # pairs of any orientation, repeated, a body with itself where radii leave
    # it out; some bodies overlap and some are in no pair
    k = rng.integers(1, max(2, int(0.9 * n) + 1), (m, 2)).astype(np.int32)
    if not with_radius and n > 1:
        same = k[:, 0] == k[:, 1]
        k[same, 1] = k[same, 1] % n + 1
    if n > 10:
        r[4] = r[5] + 1e-4 * with_radius
        r[4, 0] += 0.1 * (not with_radius)
        Gm[3] = 0.0
    rad = R if with_radius else None
    ref = O.accel_pairs(k, r, Gm, rad, acc)
    got = S.swiftest_kick_getacch_int_all_flat(n, k, r, Gm, rad, acc)
    if n == 1 and m and not with_radius:
        assert np.array_equal(ref, got, equal_nan=True)  # zero separations
    else:
        assert np.array_equal(ref.view(np.int64), got.view(np.int64))


def test_sorted_unsorted_and_unlike_separations():
    """One list three ways (sums depend on its order alone), with separations at
    the ends of the range and bodies at infinity or NaN left out by radii."""
    n, m = 60, 900
    rng, r, Gm, R, acc = _bodies(n, 5)
    r[10:14] *= 1e-130
    r[20] *= 1e130
    r[30] = np.nan
    k = rng.integers(1, n + 1, (m, 2)).astype(np.int32)
    k[k[:, 0] == k[:, 1], 1] = 1
    k = k[k[:, 0] != k[:, 1]]
    for order in (np.arange(len(k)), np.lexsort((k[:, 1], k[:, 0])), np.lexsort((k[:, 0], k[:, 1]))[::-1]):
        ref = O.accel_pairs(k[order], r, Gm, R, acc)
        got = S.swiftest_kick_getacch_int_all_flat(n, k[order], r, Gm, R, acc)
        assert np.array_equal(ref, got, equal_nan=True)


@pytest.mark.parametrize("bad", [0, -3, 41, 2**31 - 1])
def test_index_out_of_range(bad):
    n = 40
    rng, r, Gm, R, acc = _bodies(n, 6)
    k = rng.integers(1, n + 1, (500, 2)).astype(np.int32)
    k[321, rng.integers(0, 2)] = bad
    mine = acc.copy()
    rc = core.library().swg_kick_getacch_int_all_flat_pl(core.context(), n, len(k), core._c(k, np.int32), core._c(r), core._c(Gm),
                                                         core._p(R), mine)
    assert rc != 0 and np.array_equal(mine.view(np.int64), acc.view(np.int64))


def test_fast_factor():
    n, m = 500, 20000
    rng, r, Gm, R, acc = _bodies(n, 7)
    k = rng.integers(1, n + 1, (m, 2)).astype(np.int32)
    k[k[:, 0] == k[:, 1], 1] = 1
    k = k[k[:, 0] != k[:, 1]]
    acc[:] = 0.0
    ref = O.accel_pairs(k, r, Gm, None, acc)
    S.set_pair_mode(S.PAIR_FAST)
    try:
        got = S.swiftest_kick_getacch_int_all_flat(n, k, r, Gm, None, acc)
    finally:
        S.set_pair_mode(S.PAIR_EXACT)
    i, j = k[:, 0] - 1, k[:, 1] - 1
    d = np.abs(r[j] - r[i])
    w = d / ((d * d).sum(-1) ** 1.5)[:, None]
    size, count = np.zeros((n, 3)), np.bincount(np.r_[i, j], minlength=n)[:, None]
    np.add.at(size, i, Gm[j, None] * w)
    np.add.at(size, j, Gm[i, None] * w)
    # each factor within 8 ulp, one rounding a term, on both sides
    assert (np.abs(got - ref) <= 2 * (count + 8) * 2.0**-52 * size).all()
