"""Permuted copies at the edges of the tiles (32 along the source's contiguous
dim, 64 .. 512 along the last): every order of three and four dims, unit and
short dims, several blocks in one call, and the packing copy of a contraction
whose operand has no matrix form.  Copies are exact."""
import itertools

import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu

G1 = (0,)


def _tensor(rng, shapes):
    """Block i of the tensor has the shape shapes[i]; the last leg fixes the charges."""
    r, n = len(shapes[0]), len(shapes)
    t = BTensor(G1, [[s[d] for s in shapes] for d in range(r)],
                [[(i,) for i in range(n)]] + [[(0,)] * n for _ in range(r - 2)] + [[(-i,) for i in range(n)]], (0,))
    for i, s in enumerate(shapes):
        t.blocks[(i,) * r] = rng.standard_normal(s)
    return t


@pytest.mark.parametrize("perm", list(itertools.permutations(range(3))))
def test_three_dims(ctx, perm):
    rng = np.random.default_rng(1)
    t = _tensor(rng, [(1, 1, 1), (3, 5, 2), (4, 16, 7), (5, 33, 31), (17, 3, 70), (64, 4, 64), (65, 32, 65),
                      (2, 513, 5), (600, 2, 40), (33, 1, 129), (1, 40, 300)])
    out = from_dev(to_dev(ctx, t).permute(list(perm)))
    for k, b in t.blocks.items():
        assert np.array_equal(out.blocks[tuple(k[p] for p in perm)], b.transpose(perm)), b.shape


@pytest.mark.parametrize("perm", list(itertools.permutations(range(4))))
def test_four_dims(ctx, perm):
    rng = np.random.default_rng(2)
    t = _tensor(rng, [(2, 3, 4, 5), (1, 17, 1, 40), (9, 2, 33, 18), (20, 1, 6, 35), (3, 64, 2, 65)])
    out = from_dev(to_dev(ctx, t).permute(list(perm)))
    for k, b in t.blocks.items():
        assert np.array_equal(out.blocks[tuple(k[p] for p in perm)], b.transpose(perm)), b.shape


@pytest.mark.parametrize("shape", [(3, 20, 5), (40, 33, 7), (13, 70, 33), (2, 500, 12), (64, 16, 64)])
def test_packed_operand(ctx, shape):
    """Rows of dims 0 and 2 around the contracted one: packed before the product."""
    rng = np.random.default_rng(3)
    a = rng.integers(-9, 10, shape).astype(float)
    b = rng.integers(-9, 10, (shape[1], 21)).astype(float)
    A = BTensor(G1, [[s] for s in shape], [[(0,)]] * 3, (0,))
    A.blocks[(0, 0, 0)] = a
    B = BTensor(G1, [[s] for s in b.shape], [[(0,)]] * 2, (0,))
    B.blocks[(0, 0)] = b
    out = from_dev(to_dev(ctx, A).tensordot(to_dev(ctx, B), [1], [0]))
    assert np.array_equal(out.blocks[(0, 0, 0)], np.tensordot(a, b, ([1], [0])))
