"""The Gram eigensolvers at the edges of their tiles: sectors whose width is
just below, at and above a multiple of the 32-column pairs and of the 64-row
tiles, sectors of different widths in one call, spectra that end in zeros or
reach below a Gram matrix's rounding (the Cholesky factor's filled columns),
and eigh of definite, indefinite and degenerate matrices.  Values within 1e-12
of the largest (the bound the other SVD tests use: a few hundred roundings of
sums of k <= 400 terms), reconstruction within 1e-12, and the vectors of values
above 1e-10 of the largest orthonormal within 1e-12 (below, the singular values'
absolute accuracy leaves the vectors' directions open, as in the other tests)."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu

G1 = (0,)


def _diagonal(mats):
    A = BTensor(G1, [[m.shape[0] for m in mats], [m.shape[1] for m in mats]],
                [[(i,) for i in range(len(mats))], [(-i,) for i in range(len(mats))]], (0,))
    for i, m in enumerate(mats):
        A.blocks[(i, i)] = m
    return A


def _graded(rng, m, n, decades, zeros=0):
    k = min(m, n)
    u = np.linalg.qr(rng.standard_normal((m, k)))[0]
    v = np.linalg.qr(rng.standard_normal((n, k)))[0]
    s = 10.0 ** (-decades * np.arange(k) / k)
    if zeros:
        s[-zeros:] = 0.0
    return (u * s) @ v.T


@pytest.mark.parametrize("shapes,decades,zeros", [
    ([(141, 141), (160, 175)], 6, 0), ([(161, 161)], 14, 0), ([(192, 300), (30, 40), (200, 193)], 9, 0),
    ([(257, 256)], 3, 0), ([(180, 180)], 4, 60), ([(33, 33), (64, 64), (65, 65), (140, 140)], 13, 0),
    ([(32, 50), (70, 70), (139, 200)], 5, 20), ([(390, 400), (150, 150)], 8, 0)])
def test_svd_sectors_at_tile_edges(ctx, shapes, decades, zeros):
    import quantit_amd as qa
    rng = np.random.default_rng(len(shapes) * 1000 + shapes[0][0])
    mats = [_graded(rng, m, n, decades, zeros) for m, n in shapes]
    U, d, V = (from_dev(x) for x in qa.svd(to_dev(ctx, _diagonal(mats)), 1))
    for i, a in enumerate(mats):
        u, s, v = U.blocks[(i, i)], d.blocks[(i,)], V.blocks[(i, i)]
        assert np.abs(s - np.linalg.svd(a, compute_uv=False)).max() <= 1e-12 * s[0]
        assert np.linalg.norm((u * s) @ v.T - a) <= 1e-12 * np.linalg.norm(a)
        keep = s > 1e-10 * s[0]
        for w in (u[:, keep], v[:, keep]):
            assert np.abs(w.T @ w - np.eye(w.shape[1])).max() <= 1e-12


@pytest.mark.parametrize("decades,null", [(0.5, False), (12, False), (6, True)])
def test_svd_one_group_sector_widths(ctx, decades, null):
    """Every width class of the solver that takes a sector in one work-group,
    at its eight-row, register and Cholesky limits, in one call."""
    import quantit_amd as qa
    rng = np.random.default_rng(77)
    mats = [_graded(rng, k + k % 3, k, decades, k // 3 if null else 0)
            for k in (1, 2, 3, 7, 8, 9, 15, 16, 17, 25, 31, 32, 33, 47, 48, 49, 57, 63, 64, 65, 72, 73, 97)]
    U, d, V = (from_dev(x) for x in qa.svd(to_dev(ctx, _diagonal(mats)), 1))
    for i, a in enumerate(mats):
        u, s, v = U.blocks[(i, i)], d.blocks[(i,)], V.blocks[(i, i)]
        assert np.abs(s - np.linalg.svd(a, compute_uv=False)).max() <= 1e-12 * s[0]
        assert np.linalg.norm((u * s) @ v.T - a) <= 1e-12 * np.linalg.norm(a)
        keep = s > 1e-10 * s[0]
        for w in (u[:, keep], v[:, keep]):
            assert np.abs(w.T @ w - np.eye(w.shape[1])).max() <= 1e-12


@pytest.mark.parametrize("m,n,zeros", [(60, 60, 3), (200, 90, 1), (70, 150, 8)])
def test_svd_few_null_columns_are_completed(ctx, m, n, zeros):
    """Few missing directions: no unit vector lies mostly along them, and the
    null columns of U and V are orthonormal to all others all the same."""
    import quantit_amd as qa
    a = _graded(np.random.default_rng(m + n), m, n, 2, zeros)
    U, d, V = (from_dev(x) for x in qa.svd(to_dev(ctx, _diagonal([a])), 1))
    for w in (U.blocks[(0, 0)], V.blocks[(0, 0)]):
        assert np.abs(w.T @ w - np.eye(w.shape[1])).max() <= 1e-12


@pytest.mark.parametrize("k", [1, 2, 16, 33, 64, 65, 139, 140, 141, 200])
@pytest.mark.parametrize("kind", ["graded", "indefinite", "degenerate", "negative"])
def test_eigh_sector_widths(ctx, k, kind):
    import quantit_amd as qa
    rng = np.random.default_rng(k)
    q = np.linalg.qr(rng.standard_normal((k, k)))[0]
    w = {"graded": 10.0 ** (-12.0 * np.arange(k) / k), "indefinite": rng.standard_normal(k),
         "degenerate": np.repeat([2.0, -1.0, 0.5], k)[:k], "negative": -1.0 - rng.uniform(0.0, 1.0, k)}[kind]
    a = (q * w) @ q.T
    a = 0.5 * (a + a.T)
    d, U = (from_dev(x) for x in qa.eigh(to_dev(ctx, _diagonal([a])), 1))
    vals, vec = d.blocks[(0,)], U.blocks[(0, 0)]
    nrm = np.abs(w).max()
    assert np.abs(vals - np.linalg.eigvalsh(a)).max() <= 1e-12 * nrm
    assert np.abs(a @ vec - vec * vals).max() <= 1e-11 * nrm
    assert np.abs(vec.T @ vec - np.eye(k)).max() <= 1e-12


@pytest.mark.parametrize("low", [0.0, -1e-16, -1e-14, -1e-9, -1.0])
def test_eigh_around_the_definite(ctx, low):
    """Matrices just on either side of positive definite, where the solver's
    shift changes, one with zero rows among them: all in one call."""
    import quantit_amd as qa
    rng = np.random.default_rng(3)
    mats = []
    for k in (2, 7, 33, 64, 65, 130):
        q = np.linalg.qr(rng.standard_normal((k, k)))[0]
        w = 10.0 ** (-12.0 * np.arange(k) / k)
        w[k // 2:] = np.where(np.arange(k - k // 2) % 2, low, 0.0)
        a = (q * w) @ q.T
        mats.append(0.5 * (a + a.T))
    z = np.zeros((20, 20))
    z[:9, :9] = mats[1][0, 0] * np.eye(9) + 0.01
    mats.append(z)
    d, U = (from_dev(x) for x in qa.eigh(to_dev(ctx, _diagonal(mats)), 1))
    for i, a in enumerate(mats):
        vals, vec = d.blocks[(i,)], U.blocks[(i, i)]
        nrm = np.abs(a).max() * a.shape[0]
        assert np.abs(np.sort(vals) - np.linalg.eigvalsh(a)).max() <= 1e-12 * nrm
        assert np.abs(vec.T @ vec - np.eye(a.shape[0])).max() <= 1e-12
        assert np.abs(a @ vec - vec * vals).max() <= 1e-12 * nrm


# the last pass over narrow sectors is one launch up to 64 columns, 256 rows
# and 256 tiles: both sides of each limit, its quarters of 16 columns and its
# 64-row tiles, values that are zero and values that tie
@pytest.mark.parametrize("shapes,zeros", [
    ([(1, 1)], 0), ([(16, 64), (17, 65), (4, 5)], 0), ([(63, 128), (130, 64)], 2), ([(64, 256), (255, 33)], 5),
    ([(64, 257)], 0), ([(65, 65), (3, 3)], 0), ([(20, 190)] * 64, 3), ([(20, 190)] * 65, 0)])
def test_svd_narrow_sectors_at_the_last_pass(ctx, shapes, zeros):
    import quantit_amd as qa
    rng = np.random.default_rng(len(shapes) * 1000 + shapes[0][1])
    mats = [_graded(rng, m, n, 0 if i % 3 == 2 else 3, zeros) for i, (m, n) in enumerate(shapes)]
    U, d, V = (from_dev(x) for x in qa.svd(to_dev(ctx, _diagonal(mats)), 1))
    for i, a in enumerate(mats):
        u, s, v = U.blocks[(i, i)], d.blocks[(i,)], V.blocks[(i, i)]
        assert np.abs(s - np.linalg.svd(a, compute_uv=False)).max() <= 1e-12 * s[0]
        assert np.linalg.norm((u * s) @ v.T - a) <= 1e-12 * np.linalg.norm(a)
        for w in (u, v):
            assert np.abs(w.T @ w - np.eye(w.shape[1])).max() <= 1e-12


@pytest.mark.parametrize("sizes", [(1, 2, 16), (17, 48, 63, 64), (65, 7)])
def test_eigh_narrow_sectors_at_the_last_pass(ctx, sizes):
    import quantit_amd as qa
    rng = np.random.default_rng(sum(sizes))
    mats = [(lambda a: a + a.T)(rng.standard_normal((k, k))) for k in sizes]
    e, U = (from_dev(x) for x in qa.eigh(to_dev(ctx, _diagonal(mats)), 1))
    for i, a in enumerate(mats):
        w, u = e.blocks[(i,)], U.blocks[(i, i)]
        assert np.abs(w - np.linalg.eigvalsh(a)).max() <= 1e-12 * np.linalg.norm(a)
        assert np.linalg.norm((u * w) @ u.T - a) <= 1e-12 * np.linalg.norm(a)
        assert np.abs(u.T @ u - np.eye(len(w))).max() <= 1e-12


# more than eight sectors of 113 .. 140 columns stay with the solver that takes
# a sector in one work-group, up to eight take the rounds; narrower ones beside
# them stay
@pytest.mark.parametrize("count", [1, 8, 9])
@pytest.mark.parametrize("decades,zeros", [(3, 0), (12, 0), (5, 30)])
def test_svd_few_sectors_of_medium_width(ctx, count, decades, zeros):
    import quantit_amd as qa
    rng = np.random.default_rng(count * 100 + decades)
    widths = [(113, 128, 129, 140)[i % 4] for i in range(count)] + [112, 40]
    mats = [_graded(rng, k + i % 3, k + 5 * (i % 2), decades, zeros) for i, k in enumerate(widths)]
    U, d, V = (from_dev(x) for x in qa.svd(to_dev(ctx, _diagonal(mats)), 1))
    for i, a in enumerate(mats):
        u, s, v = U.blocks[(i, i)], d.blocks[(i,)], V.blocks[(i, i)]
        assert np.abs(s - np.linalg.svd(a, compute_uv=False)).max() <= 1e-12 * s[0]
        assert np.linalg.norm((u * s) @ v.T - a) <= 1e-12 * np.linalg.norm(a)
        keep = s > 1e-10 * s[0]
        for w in (u[:, keep], v[:, keep]):
            assert np.abs(w.T @ w - np.eye(w.shape[1])).max() <= 1e-12
