"""The pair tiles' test without division against the full one, at the
separations where it decides, and the per-system sums at the edges of their
chunks; the oracle's lists and states are the reference."""
import numpy as np
import pytest

import pyoracle as O
import swiftest_amd as S
from helpers import compact_disk


def _edge_pairs(seed, renc, dt, n):
    """Relative states (n, 3) around every limit of the check: separations at
    renc, at renc + |v| dt and at sqrt(2 (renc^2 + v^2 dt^2)), off by 0 to 1e-6,
    closing head on, at an angle, receding or at rest."""
    rng = np.random.Generator(np.random.PCG64(seed))
    v = renc / abs(dt) * 10.0 ** rng.uniform(-12, 8, n)
    v[rng.random(n) < 0.3] = renc / abs(dt)
    v[rng.random(n) < 0.05] = 0.0
    travel = v * abs(dt)
    lim = np.choose(rng.integers(0, 3, n), [np.full(n, renc), renc + travel, np.sqrt(2 * (renc**2 + travel**2))])
    off = np.choose(rng.integers(0, 4, n), [np.zeros(n), 10.0 ** rng.uniform(-16, -6, n), -10.0 ** rng.uniform(-16, -6, n),
                                           rng.uniform(-0.9, 1.0, n)])
    u = rng.normal(size=(n, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    w = rng.normal(size=(n, 3))
    w /= np.linalg.norm(w, axis=1)[:, None]
    mix = np.choose(rng.integers(0, 3, n), [np.zeros(n), 10.0 ** rng.uniform(-9, 0, n), np.full(n, 5.0)])[:, None]
    d = -u + mix * w
    d /= np.linalg.norm(d, axis=1)[:, None]
    return (lim * (1 + off))[:, None] * u, v[:, None] * d


def _far(x, v, renc, dt):
    """The tiles' test, the products in the kernel's order but rounded apart."""
    c2 = 2.0 * (1.0 + 1e-9)
    r2 = x[:, 0] * x[:, 0] + x[:, 1] * x[:, 1] + x[:, 2] * x[:, 2]
    v2 = v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1] + v[:, 2] * v[:, 2]
    with np.errstate(over="ignore"):
        return (r2 > c2 * dt * dt * v2 + c2 * (renc * renc)) & (r2 * v2 < 1e300)


@pytest.mark.parametrize("renc,dt", [(1.0, 0.05), (1e-4, 1.0), (1e-9, 10.0), (3e40, 1e-3), (0.5, -0.1)])
def test_far_pairs_are_never_encounters(renc, dt):
    x, v = _edge_pairs(11, renc, dt, 20000)
    z = np.zeros((1, 3))
    _, found, _ = O.encounters_pltp(z, z, x, v, np.array([renc]), dt)
    far = _far(x, v, renc, dt)
    assert far.sum() > 2000 and (~far).sum() > 2000
    assert len(found) > (500 if dt > 0 else 100) and not far[found - 1].any()


def test_far_test_at_the_ends_of_the_range():
    """Huge, infinite and NaN states: what the check accepts is never far."""
    big = [0.0, 1e-200, 1e-3, 1e75, 1e90, 1e160, np.inf, np.nan]
    x = np.array([(a, 0.0, 0.0) for a in big for _ in big])
    v = np.array([(-b, 0.0, 0.0) for _ in big for b in big])
    z = np.zeros((1, 3))
    for renc in (0.0, 1e-5, 1e80):
        for dt in (0.05, 1e-80, 1e10):
            _, found, _ = O.encounters_pltp(z, z, x, v, np.array([renc]), dt)
            with np.errstate(all="ignore"):
                assert not _far(x, v, renc, dt)[found - 1].any()


@pytest.mark.gpu
@pytest.mark.parametrize("npl,ntp", [(1, 1), (15, 63), (16, 64), (17, 65), (64, 17), (65, 300), (200, 1000), (4200, 3)])
def test_pltp_tiles(npl, ntp):
    print(f"pltp tiles {npl} x {ntp}", flush=True)
    dt, renc0 = 0.05, 1e-2
    rng = np.random.Generator(np.random.PCG64(npl + ntp))
    rp, vp = np.round(rng.normal(0, 3, (npl, 3)) * 64) / 64, np.zeros((npl, 3))
    renc = np.full(npl, renc0)
    renc[rng.random(npl) < 0.1] = 0.0
    x, v = _edge_pairs(npl, renc0, dt, ntp)
    rt = rp[rng.integers(0, npl, ntp)] + x
    ref = O.encounters_pltp(rp, vp, rt, v, renc, dt)
    got = S.encounter_check_all_pltp(npl, ntp, rp, vp, rt, v, renc, dt)
    for a, b in zip(ref, got):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 15, 17, 63, 64, 65, 129, 700])
def test_plpl_tiles(n):
    print(f"plpl tiles {n}", flush=True)
    dt, renc0 = 0.05, 1e-2
    rng = np.random.Generator(np.random.PCG64(n))
    r = np.round(rng.normal(0, 3, (n, 3)) * 64) / 64
    x, v = _edge_pairs(n, 2 * renc0, dt, n)
    v[: n // 2] = 0.0
    r[n // 2:] = r[rng.integers(0, max(n // 2, 1), n - n // 2)] + x[n // 2:]
    renc = np.full(n, renc0)
    r[0] = np.inf
    ref = O.encounters_plpl(r, v, renc, dt)
    got = S.encounter_check_all_plpl(n, r, v, renc, dt)
    for a, b in zip(ref, got):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("integ", ["HELIO", "SYMBA"])
@pytest.mark.parametrize("n", [1, 15, 16, 31, 383, 384, 385, 400, 800, 1024, 1025])
def test_sums_at_chunk_edges(integ, n):
    """Two steps (the second without vh -> vb) at the edges of the sums'
    chunks and register sets, and either side of the size up to which their
    workgroup updates the bodies, bit for bit."""
    print(f"sums {integ} {n}", flush=True)
    d = compact_disk(seed=n, npl=n, ntp=5, mlo=1e-10, mhi=1e-8)
    kind_o, kind_g = (O.HELIO, S.HELIO) if integ == "HELIO" else (O.SYMBA, S.SYMBA)
    o = O.OracleSystem(kind_o, d, 0.005, lclose=False)
    g = S.GpuSystem(kind_g, d, 0.005, lclose=False)
    for k in range(2):
        assert o.run(1) == 0
        g.run(1)
        a, b = o.state(), g.state()
        for key in ("pl_rh", "pl_vh", "pl_vb", "tp_rh", "tp_vb", "cb_vb", "ptend"):
            assert np.array_equal(np.ravel(a[key]), np.ravel(b[key])), (k, key)
