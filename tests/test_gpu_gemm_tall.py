"""Contractions whose output has more rows than 2^15 tiles of 32 or 64: whole
numbers, so every product and sum is exact.  More than 2^16 tiles of 64 are
refused."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _matrix(rng, m, n):
    A = BTensor((0,), [[m], [n]], [[(0,)], [(0,)]], (0,))
    A.blocks[(0, 0)] = rng.integers(-8, 9, (m, n)).astype(np.float64)
    return A


# 2^15 tiles of 32 are 1048576 rows, 2^16 are 2097152; 2^15 tiles of 64 2097152
@pytest.mark.parametrize("rows,n,transposed", [(1048609, 32, False), (1200000, 32, True), (2097153, 17, False)])
@pytest.mark.parametrize("variant", [None, "0", "1", "5"])
def test_tall_products_are_exact(ctx, monkeypatch, rows, n, transposed, variant):
    if variant:
        monkeypatch.setenv("QTT_GEMM_VARIANT", variant)
    rng = np.random.default_rng(rows)
    a = _matrix(rng, n, rows) if transposed else _matrix(rng, rows, n)
    b = _matrix(rng, n, n)
    d = 0 if transposed else 1
    got = from_dev(to_dev(ctx, a).tensordot(to_dev(ctx, b), [d], [0])).blocks[(0, 0)]
    x = a.blocks[(0, 0)]
    assert np.array_equal(got, (x.T if transposed else x) @ b.blocks[(0, 0)])


def test_rows_beyond_every_tile_are_refused(ctx):
    a = _matrix(np.random.default_rng(1), (1 << 22) + 1, 1)
    b = _matrix(np.random.default_rng(2), 1, 17)
    with pytest.raises(ValueError, match="rows or columns"):
        to_dev(ctx, a).tensordot(to_dev(ctx, b), [1], [0])


@pytest.mark.parametrize("rows", [(1 << 19) - 1, 1 << 19, (1 << 19) + 1, (1 << 20) + 129, 3000000])
@pytest.mark.parametrize("k,n,transposed", [(2, 3, False), (16, 5, True), (17, 5, False)])
def test_tall_narrow_products_are_exact(ctx, rows, k, n, transposed):
    """Tasks of several 128 rows from 2^19 rows on, up to K = 16."""
    rng = np.random.default_rng(rows)
    a, b = _matrix(rng, *((k, rows) if transposed else (rows, k))), _matrix(rng, k, n)
    got = from_dev(to_dev(ctx, a).tensordot(to_dev(ctx, b), [0 if transposed else 1], [0])).blocks[(0, 0)]
    x = a.blocks[(0, 0)]
    assert np.array_equal(got, (x.T if transposed else x) @ b.blocks[(0, 0)])


def test_many_tall_narrow_blocks_are_exact(ctx):
    """Blocks of a few rows to 300000 beside each other in tasks of 256 rows."""
    rng = np.random.default_rng(3)
    rows = [1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300000, 300001]
    A = BTensor((0,), [rows, [2] * len(rows)], [[(i,) for i in range(len(rows))], [(-i,) for i in range(len(rows))]], (0,))
    for i, m in enumerate(rows):
        A.blocks[(i, i)] = rng.integers(-8, 9, (m, 2)).astype(float)
    C = BTensor((0,), [[2] * len(rows), [3] * len(rows)],
                [[(i,) for i in range(len(rows))], [(-i,) for i in range(len(rows))]], (0,))
    for i in range(len(rows)):
        C.blocks[(i, i)] = rng.integers(-8, 9, (2, 3)).astype(float)
    got = from_dev(to_dev(ctx, A).tensordot(to_dev(ctx, C), [1], [0]))
    for i in range(len(rows)):
        assert np.array_equal(got.blocks[(i, i)], A.blocks[(i, i)] @ C.blocks[(i, i)])
