"""The global cut where the number of singular values lies around the limits
of its two sorts, with values that tie across sectors: kept counts are those
of the oracle exactly."""
import numpy as np
import pytest

import oracle.btensor_oracle as bo
from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("total", [1, 2, 3, 63, 64, 65, 255, 256, 257, 500, 511, 512, 513, 700])
@pytest.mark.parametrize("max_size,tol", [(2 ** 62, 1e-2), (37, 0.0), (2 ** 62, 0.0)])
def test_cut_at_the_sort_limits(ctx, total, max_size, tol):
    import quantit_amd as qa
    rng = np.random.default_rng(total)
    sizes = []
    while sum(sizes) < total:
        sizes.append(min(int(rng.integers(1, 41)), total - sum(sizes)))
    n = len(sizes)
    t = BTensor((0,), [sizes, sizes], [[(i,) for i in range(n)], [(-i,) for i in range(n)]], (0,))
    levels = 2.0 ** -np.arange(12)  # ties within and across sectors, exact in every step
    for i, k in enumerate(sizes):
        t.blocks[(i, i)] = np.diag(rng.choice(levels, k))
    _, d, _ = (from_dev(x) for x in qa.svd(to_dev(ctx, t), 1, tol=tol, min_size=1, max_size=max_size))
    _, want, _ = bo.svd_truncated(t, 1, tol, 1, max_size)
    assert sorted(d.blocks) == sorted(want.blocks)
    for k in want.blocks:
        assert np.array_equal(d.blocks[k], want.blocks[k])
