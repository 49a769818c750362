"""Launch descriptors on both sides of the limits at which they travel in the
kernel's arguments, in a runtime copy and in a copy kernel: many small blocks,
so that the lists are long and the data is not.  Integers: every result is
exact."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu

G1 = (0,)


def _tensor(rng, blocks, charge=1, size=2):
    t = BTensor(G1, [[size] * blocks, [size + 1] * blocks], [[(charge * i,) for i in range(blocks)],
                                                            [(-charge * i,) for i in range(blocks)]], (0,))
    for i in range(blocks):
        t.blocks[(i, i)] = rng.integers(-9, 10, (size, size + 1)).astype(float)
    return t


# 40, 32, 32 and about 100 bytes a block: 3584 and 16384 bytes lie between
@pytest.mark.parametrize("blocks", [1, 33, 34, 35, 36, 37, 74, 75, 89, 90, 99, 100, 112, 113, 150, 170, 341, 342, 410,
                                    411, 512, 513, 2000])
def test_every_operation_at_the_list_limits(ctx, blocks):
    rng = np.random.default_rng(blocks)
    a, b = _tensor(rng, blocks), _tensor(rng, blocks)
    da, db = to_dev(ctx, a), to_dev(ctx, b)
    flat = [(a.blocks[(i, i)], b.blocks[(i, i)]) for i in range(blocks)]
    added = from_dev(da.add(db, 3.0))
    turned = from_dev(da.permute([1, 0]))
    prod = from_dev(da.tensordot(to_dev(ctx, _tensor(np.random.default_rng(1), blocks, -1)), [0], [0]))
    other = _tensor(np.random.default_rng(1), blocks, -1)
    for i, (x, y) in enumerate(flat):
        assert np.array_equal(added.blocks[(i, i)], x + 3.0 * y)
        assert np.array_equal(turned.blocks[(i, i)], x.T)
        assert np.array_equal(prod.blocks[(i, i)], x.T @ other.blocks[(i, i)])
    assert da.full_dot(db) == sum(float((x * y).sum()) for x, y in flat)
