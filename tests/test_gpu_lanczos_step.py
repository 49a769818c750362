"""The Lanczos step in one launch against exact diagonalisation: vectors of
each width class (at full bond the two-site space of the middle bond is the
whole charge sector: 252, 924, 3432 states) with few and many Krylov vectors,
and of more than 8192 elements at the last, where the steps of wide bonds go in
launches over all CUs and those of the others in one.  A converged solve's energy
is the lowest eigenvalue; the bound is the other solves' 1e-10."""
import itertools

import numpy as np
import pytest

from oracle import dmrg_oracle as dor
from tests.helpers import to_dev
from tests.test_gpu_dmrg import _lanczos_ctx, _setup

pytestmark = pytest.mark.gpu


def _exact(L, delta, fields):
    """Lowest eigenvalue of the chain with as many spins up as down."""
    from scipy.sparse import coo_matrix
    from scipy.sparse.linalg import eigsh
    states = [sum(1 << i for i in c) for c in itertools.combinations(range(L), L // 2)]
    index = {s: i for i, s in enumerate(states)}
    rows, cols, vals = [], [], []
    for k, s in enumerate(states):
        sz = [0.5 if s >> i & 1 else -0.5 for i in range(L)]
        rows.append(k)
        cols.append(k)
        vals.append(delta * sum(sz[i] * sz[i + 1] for i in range(L - 1)) + sum(f * z for f, z in zip(fields, sz)))
        for i in range(L - 1):
            if sz[i] != sz[i + 1]:
                rows.append(k)
                cols.append(index[s ^ (3 << i)])
                vals.append(0.5)
    h = coo_matrix((vals, (rows, cols))).tocsr()
    return eigsh(h, k=1, which="SA", tol=0)[0][0]


@pytest.mark.parametrize("L,bond,krylov", [(10, 32, 4), (12, 64, 9), (14, 128, 6), (14, 128, 40), (16, 256, 8)])
def test_converged_solve_is_exact(ctx, L, bond, krylov):
    import quantit_amd as qa
    rng = np.random.default_rng(L + krylov)
    fields = rng.uniform(-1.0, 1.0, L)
    mpo, mps = _setup(dor.xxz_field_dense(0.7, fields), seed=6)
    opts = qa.DmrgOptions(cutoff=1e-14, convergence_criterion=1e-13, maximum_bond=bond, minimum_bond=4,
                          maximum_iterations=12)
    with _lanczos_ctx(ctx, krylov, 1e-14):
        E, _, _ = qa.dmrg([to_dev(ctx, t) for t in mpo], [to_dev(ctx, t) for t in mps], opts)
    # all-up is either of the two spin directions: the fields' sign
    e0 = min((_exact(L, 0.7, f) for f in (fields, -fields)), key=lambda e: abs(e - E))
    assert abs(E - e0) <= 1e-10 * abs(e0)
