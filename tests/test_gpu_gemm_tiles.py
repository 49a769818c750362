"""The grouped FP64 GEMM at the edges of its tiles and k steps, for every way
the operands can be contiguous, both tile sizes and the general kernel.
Entries are small integers, so every sum is exact and the result must equal
numpy's bit for bit; entries next to the operands in memory are infinite
nowhere but in one case, which must not leak in from rows or k past an edge."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu

G1 = (0,)
SIZES = [(1, 1, 1), (1, 40, 2), (33, 1, 15), (31, 32, 16), (32, 33, 17), (63, 64, 31), (64, 65, 32), (65, 63, 33),
         (2, 130, 100), (129, 3, 64), (96, 96, 1), (17, 200, 5)]


def _diag(mats):
    t = BTensor(G1, [[m.shape[0] for m in mats], [m.shape[1] for m in mats]],
                [[(i,) for i in range(len(mats))], [(-i,) for i in range(len(mats))]], (0,))
    for i, m in enumerate(mats):
        t.blocks[(i, i)] = m
    return t


@pytest.mark.parametrize("variant", ["0", "1", "5"])
@pytest.mark.parametrize("da,db", [(1, 0), (1, 1), (0, 0), (0, 1)])
def test_tiles_and_layouts_are_exact(ctx, monkeypatch, variant, da, db):
    monkeypatch.setenv("QTT_GEMM_VARIANT", variant)
    monkeypatch.setenv("QTT_GEMM_ROWS", "0")
    rng = np.random.default_rng(10 * da + db)
    a = [rng.integers(-9, 10, (m, k) if da == 1 else (k, m)).astype(float) for m, n, k in SIZES]
    b = [rng.integers(-9, 10, (k, n) if db == 0 else (n, k)).astype(float) for m, n, k in SIZES]
    A, B = _diag(a), _diag(b)
    if da == db:  # the contracted legs' charges have to cancel
        B.cvals = [[tuple(-x for x in c) for c in leg] for leg in B.cvals]
    out = from_dev(to_dev(ctx, A).tensordot(to_dev(ctx, B), [da], [db]))
    for i in range(len(SIZES)):
        x = a[i] if da == 1 else a[i].T
        y = b[i] if db == 0 else b[i].T
        assert np.array_equal(out.blocks[(i, i)], x @ y), SIZES[i]


@pytest.mark.parametrize("variant", ["1", "5"])
def test_values_past_an_edge_stay_out(ctx, monkeypatch, variant):
    """The neighbours of a block in memory are infinite: rows and k beyond the
    block's edges must not reach its result."""
    monkeypatch.setenv("QTT_GEMM_VARIANT", variant)
    monkeypatch.setenv("QTT_GEMM_ROWS", "0")
    rng = np.random.default_rng(5)
    inf = np.full((20, 20), np.inf)
    a = [inf, rng.integers(-9, 10, (37, 21)).astype(float), inf]
    b = [inf, rng.integers(-9, 10, (21, 43)).astype(float), inf]
    out = from_dev(to_dev(ctx, _diag(a)).tensordot(to_dev(ctx, _diag(b)), [1], [0]))
    assert np.array_equal(out.blocks[(1, 1)], a[1] @ b[1])


@pytest.mark.parametrize("variant", ["1", "5"])
def test_pairs_without_a_common_layout(ctx, monkeypatch, variant):
    """Sections of one beside wider ones over two contracted legs: the blocks'
    matrix views are contiguous in different dimensions."""
    monkeypatch.setenv("QTT_GEMM_VARIANT", variant)
    monkeypatch.setenv("QTT_GEMM_ROWS", "0")
    rng = np.random.default_rng(6)
    l, s, w = [(5, (0,)), (1, (1,))], [(1, (0,)), (3, (1,))], [(2, (0,)), (1, (-1,)), (4, (-2,))]
    inv = lambda leg: [(n, tuple(-x for x in c)) for n, c in leg]  # noqa: E731
    A = BTensor.from_sections(G1, [l, s, w], (0,))
    B = BTensor.from_sections(G1, [inv(w), inv(l), inv(s)], (0,))
    for t in (A, B):
        for idx in t.all_allowed_indices():
            t.blocks[idx] = rng.integers(-9, 10, t.block_shape(idx)).astype(float)
    for da, db in (([0], [1]), ([1], [2]), ([2], [0]), ([0, 1], [1, 2]), ([1, 0], [2, 1]), ([2, 0], [0, 1])):
        out = from_dev(to_dev(ctx, A).tensordot(to_dev(ctx, B), da, db))
        ref = np.tensordot(A.to_dense(), B.to_dense(), (da, db))
        assert np.array_equal(out.to_dense(), ref), (da, db)


@pytest.mark.parametrize("rows", [1, 15, 17, 64, 65, 129, 40_000])
def test_narrow_products_are_exact(ctx, rows):
    """The row kernel: several pairs to an output, summed K over no whole
    chunks of four, every column count, both task sizes (the last entry has
    more than 2^17 rows in all); infinite neighbours stay out."""
    rng = np.random.default_rng(rows)
    for ks, cols in (([1], [1, 2]), ([1, 2, 2], [3, 4, 5, 16]), ([5, 60, 63], [7, 12])):
        m = [rows, 1 + rows // 2]
        A = BTensor(G1, [m, ks], [[(0,)] * len(m), [(0,)] * len(ks)], (0,))
        B = BTensor(G1, [ks, cols], [[(0,)] * len(ks), [(0,)] * len(cols)], (0,))
        for i, r in enumerate(m):
            for j, k in enumerate(ks):
                A.blocks[(i, j)] = rng.integers(-9, 10, (r, k)).astype(float)
        for j, k in enumerate(ks):
            for i, n in enumerate(cols):
                B.blocks[(j, i)] = rng.integers(-9, 10, (k, n)).astype(float)
        inf = np.inf
        A.blocks[(1, len(ks) - 1)][:] = inf  # reaches the second row block only
        out = from_dev(to_dev(ctx, A).tensordot(to_dev(ctx, B), [1], [0]))
        for c in range(len(cols)):
            ref = sum(A.blocks[(0, j)] @ B.blocks[(j, c)] for j in range(len(ks)))
            assert np.array_equal(out.blocks[(0, c)], ref), (ks, cols[c])
