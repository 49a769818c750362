"""Elementwise passes, dot products and the sums of split products where a
block ends around a wave, a workgroup and a workgroup's 2048 elements.
Integers: every result is exact."""
import numpy as np
import pytest

import oracle.btensor_oracle as bo
from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _tensor(rng, dims):
    t = BTensor((0,), [[d] for d in dims], [[(0,)] for _ in dims], (0,))
    t.blocks[(0,) * len(dims)] = rng.integers(1, 10, dims).astype(float)
    return t


@pytest.mark.parametrize("dims", [(1, 1), (1, 63), (5, 51), (16, 16), (257, 1), (23, 89), (2, 1024), (683, 3), (45, 91),
                                  (4096, 1), (1, 4097), (131, 513)])
def test_elementwise_and_dot(ctx, dims):
    rng = np.random.default_rng(dims[0] * 10007 + dims[1])
    a, b, last, one = _tensor(rng, dims), _tensor(rng, dims), _tensor(rng, dims[1:]), _tensor(rng, ())
    x, y, da, db = a.blocks[(0, 0)], b.blocks[(0, 0)], to_dev(ctx, a), to_dev(ctx, b)
    got = lambda t: from_dev(t).blocks[(0, 0)]
    assert np.array_equal(got(da.add(db, -2.0)), x - 2.0 * y)
    assert np.array_equal(got(da.mul(db)), x * y)
    assert np.array_equal(got(da.mul(to_dev(ctx, last))), x * last.blocks[(0,)])
    assert np.array_equal(got(da.mul(to_dev(ctx, one))), x * one.blocks[()])
    assert np.array_equal(got(da.permute([1, 0])), x.T)
    assert da.full_dot(db) == float((x * y).sum())


@pytest.mark.parametrize("m,n,k", [(1, 1, 40000), (30, 40, 20000), (45, 46, 9000), (64, 65, 8192)])
def test_sums_of_split_products(ctx, m, n, k):
    rng = np.random.default_rng(m)
    a, b = _tensor(rng, (k, m)), _tensor(rng, (k, n))
    got = from_dev(to_dev(ctx, a).tensordot(to_dev(ctx, b), [0], [0]))
    assert np.array_equal(got.blocks[(0, 0)], bo.tensordot(a, b, [0], [0]).blocks[(0, 0)])


# blocks that only one operand has break a run, at its ends and inside
@pytest.mark.parametrize("has_x,has_y", [("11111111", "11111111"), ("11111111", "01111110"), ("10110111", "11101101"),
                                         ("10101010", "01010101"), ("00001111", "11111111"), ("10000000", "00000001")])
@pytest.mark.parametrize("size", [(3, 2), (40, 30)])
def test_runs_of_blocks(ctx, has_x, has_y, size):
    rng = np.random.default_rng(int(has_x, 2) * 256 + int(has_y, 2))
    ops = []
    for has in (has_x, has_y):
        t = BTensor((0,), [[size[0]] * 8, [size[1]] * 8], [[(i,) for i in range(8)], [(-i,) for i in range(8)]], (0,))
        for i in range(8):
            if has[i] == "1":
                t.blocks[(i, i)] = rng.integers(-9, 10, size).astype(float)
        ops.append(t)
    x, y = ops
    one = _tensor(rng, ())
    dx, dy, done = to_dev(ctx, x), to_dev(ctx, y), to_dev(ctx, one)
    for got, want in [(dx.add(dy, 3.0), bo.add(x, y, 3.0)), (dx.mul(dy), bo.mul(x, y)), (dx.mul(done), bo.mul(x, one))]:
        got = from_dev(got)
        assert sorted(got.blocks) == sorted(want.blocks)
        assert all(np.array_equal(got.blocks[k], want.blocks[k]) for k in want.blocks)
    assert dx.full_dot(dy) == sum(float((x.blocks[k] * y.blocks[k]).sum()) for k in x.blocks if k in y.blocks)
