"""SVD of matrices of lower rank, plain or behind a spectrum of many decades.
Singular values within 1e-14 of the largest, zeros included: the input's
rounding is about sqrt(k) eps = 4e-15 of it at 300 columns, and every step is an
orthogonal transform.  All columns of U and V orthonormal to 1e-12, the product
within 1e-12 of the norm, as in the other tests."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _sector(m):
    A = BTensor((0,), [[m.shape[0]], [m.shape[1]]], [[(0,)], [(0,)]], (0,))
    A.blocks[(0, 0)] = m
    return A


def _matrix(m, k, s, seed=5):
    rng = np.random.default_rng(seed)
    u = np.linalg.qr(rng.standard_normal((m, k)))[0]
    return (u * s) @ np.linalg.qr(rng.standard_normal((k, k)))[0].T


def _svd(ctx, a):
    import quantit_amd as qa
    U, d, V = (from_dev(x) for x in qa.svd(to_dev(ctx, _sector(a)), 1))
    u, s, v = U.blocks[(0, 0)], d.blocks[(0,)], V.blocks[(0, 0)]
    assert np.linalg.norm((u * s) @ v.T - a) <= 1e-12 * np.linalg.norm(a)
    return u, s, v


@pytest.mark.parametrize("m,k", [(24, 24), (64, 64), (100, 100), (400, 130), (160, 160), (300, 300)])
@pytest.mark.parametrize("kind", ["a quarter", "ten", "half of ten decades"])
def test_null_values_and_vectors(ctx, m, k, kind):
    x = np.arange(k)
    s = {"a quarter": np.where(x < k // 4, 1.0 + x / k, 0.0), "ten": np.where(x < 10, 1.0 + x / k, 0.0),
         "half of ten decades": np.where(x < k // 2, 10.0 ** (-20.0 * x / k), 0.0)}[kind]
    u, got, v = _svd(ctx, _matrix(m, k, s))
    assert np.abs(got - np.sort(s)[::-1]).max() <= 1e-14 * s.max()
    for w in (u, v):
        assert np.abs(w.T @ w - np.eye(k)).max() <= 1e-12


@pytest.mark.parametrize("m,k", [(24, 24), (64, 64), (400, 130), (160, 160), (300, 300)])
@pytest.mark.parametrize("decades", [20, 30])
def test_spectra_below_the_rounding(ctx, m, k, decades):
    """The Gram iterations converge: V is the product of two to four orthogonal
    factors, each within sqrt(k) roundings of one."""
    import quantit_amd as qa
    s = 10.0 ** (-decades * np.arange(k) / k)
    own = qa.Context(0, arena_bytes=256 << 20)
    u, got, v = _svd(own, _matrix(m, k, s))
    assert own.svd_stats()["max_sweeps"] <= 5
    own.close()
    assert np.abs(got - s).max() <= 1e-14
    assert np.abs(v.T @ v - np.eye(k)).max() <= 4 * np.sqrt(k) * 2.3e-16 + 1e-14
    keep = got > 1e-10
    assert np.abs(u[:, keep].T @ u[:, keep] - np.eye(keep.sum())).max() <= 1e-12
