"""eigh and SVD of sectors whose columns do not all couple (hidden symmetries,
direct sums): in the one-work-group solver eight lanes rotate a pair, the eight
pairs of a wave independently of each other, and a sweep may only be the last
when no pair of any of them rotated far.  Vectors orthonormal, values and
residuals within 1e-12 of the norm (the bound of the other eigensolver tests)."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _sector(m):
    A = BTensor((0,), [[m.shape[0]], [m.shape[1]]], [[(0,)], [(0,)]], (0,))
    A.blocks[(0, 0)] = m
    return A


def _matrix(kind, k):
    """A positive definite k x k matrix."""
    if kind == "random beside a lone state":
        x = np.random.default_rng(k).standard_normal((k - 1, k - 1))
        g = np.zeros((k, k))
        g[0, 0] = 10.0 * k
        g[1:, 1:] = x @ x.T + np.eye(k - 1)
        return g
    # diagonals that fall so evenly that pivoting keeps the order, column c
    # coupled to c + 8 in every sixteen
    d = 2.0 - 0.05 * np.arange(k) if kind == "even steps" else 2.0 ** (-0.2 * np.arange(k))
    g = np.diag(d)
    for c in range(k - 8):
        if c // 8 % 2 == 0 and (kind == "all in pairs" or c % 8):
            g[c, c + 8] = g[c + 8, c] = 0.3 if kind == "even steps" else 0.3 * np.sqrt(d[c] * d[c + 8])
    return g


CASES = [("even steps", 16)] + [(kind, k) for kind in ("first of eight alone", "all in pairs",
                                                       "random beside a lone state") for k in (16, 32, 64, 130)]


@pytest.mark.parametrize("kind,k", CASES)
def test_eigh_of_decoupled_columns(ctx, kind, k):
    import quantit_amd as qa
    g = _matrix(kind, k)
    e, U = (from_dev(x) for x in qa.eigh(to_dev(ctx, _sector(g)), 1))
    w, u = e.blocks[(0,)], U.blocks[(0, 0)]
    nrm = np.linalg.norm(g, 2)
    assert np.abs(u.T @ u - np.eye(k)).max() <= 1e-12
    assert np.abs(w - np.linalg.eigvalsh(g)).max() <= 1e-12 * nrm
    assert np.abs(g @ u - u * w).max() <= 1e-12 * nrm


@pytest.mark.parametrize("kind,k", CASES)
def test_svd_of_decoupled_columns(ctx, kind, k):
    import quantit_amd as qa
    g = _matrix(kind, k)
    q = np.linalg.qr(np.random.default_rng(k).standard_normal((k + 5, k)))[0]
    a = q @ np.linalg.cholesky(g).T  # a^T a = g
    U, d, V = (from_dev(x) for x in qa.svd(to_dev(ctx, _sector(a)), 1))
    u, s, v = U.blocks[(0, 0)], d.blocks[(0,)], V.blocks[(0, 0)]
    for w in (u, v):
        assert np.abs(w.T @ w - np.eye(k)).max() <= 1e-12
    assert np.abs(s - np.linalg.svd(a, compute_uv=False)).max() <= 1e-12 * s[0]
    assert np.linalg.norm((u * s) @ v.T - a) <= 1e-12 * np.linalg.norm(a)


@pytest.mark.parametrize("precond", ["0", "1"])
@pytest.mark.parametrize("k", [2, 16, 65, 130])
def test_eigh_of_indefinite_matrices_with_a_positive_diagonal(ctx, k, precond, monkeypatch):
    """Nothing but the factorisation shows that these are not definite, and
    QTT_SVD_PRECOND=0 does without it."""
    import quantit_amd as qa
    monkeypatch.setenv("QTT_SVD_PRECOND", precond)
    x = np.random.default_rng(k).uniform(-1.0, 1.0, (k, k))
    g = x + x.T
    np.fill_diagonal(g, 0.5)
    g[0, 1] = g[1, 0] = 0.8
    e, U = (from_dev(x) for x in qa.eigh(to_dev(ctx, _sector(g)), 1))
    w, u = e.blocks[(0,)], U.blocks[(0, 0)]
    nrm = np.linalg.norm(g)
    assert w[0] < 0.0
    assert np.abs(w - np.linalg.eigvalsh(g)).max() <= 1e-12 * nrm
    assert np.abs(g @ u - u * w).max() <= 1e-12 * nrm
    assert np.abs(u.T @ u - np.eye(k)).max() <= 1e-12


@pytest.mark.parametrize("coupling", [0.0, 1e-13, 1e-3])
def test_eigh_of_wide_almost_diagonal_matrices(ctx, coupling):
    """A wide sector that is diagonal to the rounding is not factored, whatever
    the one beside it; couplings above the rounding are solved."""
    import quantit_amd as qa
    rng = np.random.default_rng(9)
    x = rng.standard_normal((150, 150))
    mats = [np.diag(rng.uniform(-1.0, 1.0, 200)), np.diag(np.full(141, 2.0)), x + x.T]
    y = rng.standard_normal((200, 200))
    mats[0] += coupling * (y + y.T)
    A = BTensor((0,), [[200, 141, 150]] * 2, [[(0,), (1,), (2,)], [(0,), (-1,), (-2,)]], (0,))
    for i, m in enumerate(mats):
        A.blocks[(i, i)] = m
    capped = ctx.svd_stats()["unconverged"]
    e, U = (from_dev(x) for x in qa.eigh(to_dev(ctx, A), 1))
    assert ctx.svd_stats()["unconverged"] == capped
    for i, a in enumerate(mats):
        w, u, nrm = e.blocks[(i,)], U.blocks[(i, i)], np.linalg.norm(a)
        assert np.abs(w - np.linalg.eigvalsh(a)).max() <= 1e-12 * nrm
        assert np.abs(a @ u - u * w).max() <= 1e-13 * nrm
        assert np.abs(u.T @ u - np.eye(len(a))).max() <= 1e-12
    del A.blocks[(2, 2)]
    ctx.set_profiling(True)
    ctx.kernel_times()
    qa.eigh(to_dev(ctx, A), 1)
    names = ctx.kernel_times()
    ctx.set_profiling(False)
    assert ("svd_pchol" in names) == (coupling > 0.0)


def test_eigh_counts_its_sweeps():
    """The largest sweep count of a call: the sweeps over a wide sector, none of
    those that one work-group makes."""
    import quantit_amd as qa
    ctx = qa.Context(0, arena_bytes=256 << 20)
    for k, sweeps in ((60, range(0, 1)), (200, range(3, 30))):
        x = np.random.default_rng(k).standard_normal((k, k))
        qa.eigh(to_dev(ctx, _sector(x + x.T)), 1)
        assert ctx.svd_stats()["max_sweeps"] in sweeps
    ctx.close()
