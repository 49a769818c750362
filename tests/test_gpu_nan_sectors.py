"""Decompositions of matrices that hold a NaN or an infinity return: some of the
sector's values are not finite, its neighbours' are as they are without it."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _pair(bad):
    good = np.diag(np.arange(1.0, 6.0)) + 0.1
    A = BTensor((0,), [[len(bad), 5]] * 2, [[(0,), (1,)], [(0,), (-1,)]], (0,))
    A.blocks[(0, 0)], A.blocks[(1, 1)] = bad, good
    return A, good


def _spoiled(k, where, value):
    x = np.random.default_rng(k).standard_normal((k, k))
    m = x @ x.T + k * np.eye(k)
    i, j = {"diagonal": (k // 2, k // 2), "beside": (0, k - 1)}[where]
    m[i, j] = m[j, i] = value
    return m


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("where", ["diagonal", "beside"])
@pytest.mark.parametrize("k", [2, 16, 64, 65, 140, 141])
def test_eigh_returns(ctx, k, where, value):
    import quantit_amd as qa
    A, good = _pair(_spoiled(k, where, value))
    e, U = (from_dev(x) for x in qa.eigh(to_dev(ctx, A), 1))
    assert not np.isfinite(e.blocks[(0,)]).all()
    assert np.abs(e.blocks[(1,)] - np.linalg.eigvalsh(good)).max() <= 1e-12 * np.linalg.norm(good)
