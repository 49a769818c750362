"""Decompositions in an arena that holds the input, the result and the rounds'
work matrices but not the Gram iterations': they go by the rounds alone.  The
arenas are what the calls needed before eigh and the wide sectors' sweeps took
buffers of their own, and a little; that of the last SVD is smaller."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _context(megabytes):
    """An arena with that much beside the staging ring (a quarter, 1 MB at least)."""
    import quantit_amd as qa
    x = megabytes * 1e6
    return qa.Context(0, arena_bytes=int(x + max(1 << 20, x / 3)))


def _sectors(mats):
    n = len(mats)
    A = BTensor((0,), [[m.shape[0] for m in mats], [m.shape[1] for m in mats]],
                [[(i,) for i in range(n)], [(-i,) for i in range(n)]], (0,))
    for i, m in enumerate(mats):
        A.blocks[(i, i)] = m
    return A


# input + measured need, in MB
@pytest.mark.parametrize("k,count,arena", [(60, 20, 0.6 + 2.1), (140, 1, 0.2 + 0.7), (300, 1, 0.8 + 3.3)])
def test_eigh(k, count, arena):
    import quantit_amd as qa
    ctx = _context(arena)
    rng = np.random.default_rng(k)
    mats = [x + x.T for x in rng.standard_normal((count, k, k))]
    e, U = (from_dev(x) for x in qa.eigh(to_dev(ctx, _sectors(mats)), 1))
    for i, a in enumerate(mats):
        w, u, nrm = e.blocks[(i,)], U.blocks[(i, i)], np.linalg.norm(a, 2)
        assert np.abs(w - np.linalg.eigvalsh(a)).max() <= 1e-12 * nrm
        assert np.abs(a @ u - u * w).max() <= 1e-12 * nrm
        assert np.abs(u.T @ u - np.eye(k)).max() <= 1e-12
    ctx.close()


@pytest.mark.parametrize("m,n,arena", [(130, 130, 0.2 + 1.5), (160, 160, 0.3 + 2.3), (600, 600, 2.9 + 33.5),
                                       (300, 300, 0.8 + 4.5)])
def test_svd(m, n, arena):
    import quantit_amd as qa
    ctx = _context(arena)
    a = np.random.default_rng(m).standard_normal((m, n))
    U, d, V = (from_dev(x) for x in qa.svd(to_dev(ctx, _sectors([a])), 1))
    u, s, v = U.blocks[(0, 0)], d.blocks[(0,)], V.blocks[(0, 0)]
    assert np.abs(s - np.linalg.svd(a, compute_uv=False)).max() <= 1e-12 * s[0]
    assert np.linalg.norm((u * s) @ v.T - a) <= 1e-12 * np.linalg.norm(a)
    for w in (u, v):
        assert np.abs(w.T @ w - np.eye(w.shape[1])).max() <= 1e-12
    ctx.close()
