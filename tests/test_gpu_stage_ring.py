"""Descriptor lists longer than the staging ring, and rings that wrap within a
call: a context with a ring of 64 KB (QTT_STAGE_BYTES) gives the same bits as
one with the usual 64 MB."""
import numpy as np
import pytest

from oracle.btensor_oracle import BTensor
from tests.helpers import from_dev, rand_btensor, rand_leg, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture
def small(monkeypatch):
    import quantit_amd as qa
    monkeypatch.setenv("QTT_STAGE_BYTES", str(64 << 10))
    c = qa.Context(0, arena_bytes=2 << 30)
    yield c
    c.close()


def _same(x, y):
    assert sorted(x.blocks) == sorted(y.blocks)
    for k in y.blocks:
        assert np.array_equal(x.blocks[k], y.blocks[k]), k


def _one_block(*dims):
    A = BTensor((0,), [[d] for d in dims], [[(0,)] for _ in dims], (0,))
    A.blocks[(0,) * len(dims)] = np.random.default_rng(sum(dims)).standard_normal(dims)
    return A


@pytest.mark.parametrize("dims", [(20000, 32, 32), (60000, 3, 101)])
def test_permute(ctx, small, dims):
    a = _one_block(*dims)  # more than 8192 tasks of 8 bytes
    got = from_dev(to_dev(small, a).permute([0, 2, 1]))
    assert np.array_equal(got.blocks[(0, 0, 0)], a.blocks[(0, 0, 0)].transpose(0, 2, 1))


def test_contraction_with_packed_operands(ctx, small):
    a, b = _one_block(500, 300, 64), _one_block(300, 200)
    ref, got = (from_dev(to_dev(c, a).tensordot(to_dev(c, b), [1], [0])) for c in (ctx, small))
    _same(got, ref)


def test_contraction_of_many_blocks(ctx, small):
    rng = np.random.default_rng(5)
    l, r = rand_leg(rng, 40, -20, 20, 1, 6), rand_leg(rng, 40, -20, 20, 1, 30)
    s = [(2, (q,)) for q in range(-6, 7)]
    inv = [(n, (-q[0],)) for n, q in r]
    a, b = rand_btensor(rng, (0,), [l, s, r], (0,)), rand_btensor(rng, (0,), [inv, s, l], (0,))
    ref, got = (from_dev(to_dev(c, a).tensordot(to_dev(c, b), [2], [0])) for c in (ctx, small))
    _same(got, ref)


def test_svd_of_wide_sectors(ctx, small):
    """The rounds' work items alone are longer than the ring."""
    import quantit_amd as qa
    rng = np.random.default_rng(6)
    shapes = [(600, 600), (500, 700), (300, 300), (310, 290), (130, 160), (40, 40)]
    A = BTensor((0,), [[m for m, _ in shapes], [n for _, n in shapes]],
                [[(i,) for i in range(len(shapes))], [(-i,) for i in range(len(shapes))]], (0,))
    for i, (m, n) in enumerate(shapes):
        A.blocks[(i, i)] = rng.standard_normal((m, n))
    for ref, got in zip(*([from_dev(x) for x in qa.svd(to_dev(c, A), 1)] for c in (ctx, small))):
        _same(got, ref)


def test_dmrg(ctx, small):
    import quantit_amd as qa
    from oracle import dmrg_oracle as dor
    mpo = dor.guess_bmpo(dor.drop_zero_channels(dor.xxz_field_dense(0.8, np.linspace(-1, 1, 10))),
                         dor.u1_spin_half_phys())
    mps = dor.prepare_state(dor.random_bmps(8, mpo, (0,), 2))
    E = [qa.dmrg([to_dev(c, t) for t in mpo], [to_dev(c, t) for t in mps],
                 qa.DmrgOptions(cutoff=1e-8, convergence_criterion=0.0, maximum_bond=24, maximum_iterations=4))[0]
         for c in (ctx, small)]
    assert E[0] == E[1]


@pytest.mark.parametrize("j,k", [(32, 64), (20, 40), (4, 16)])
def test_allocation_free_contraction_that_fills_128_mib(ctx, j, k):
    """A packed operand that leaves 100 KB of 128 MiB to the lists, however
    finely the copy and the rows are divided."""
    import quantit_amd as qa
    i = ((128 << 20) - 100000) // 8 // (j * k)
    rng = np.random.default_rng(j)
    x, v = rng.integers(-8, 9, (i, k, j)).astype(float), rng.integers(-8, 9, (k, 3)).astype(float)
    a = qa.BTensor.from_parts(ctx, (0,), [[i], [k], [j]], [[(0,)]] * 3, (0,), {(0, 0, 0): x})
    b = qa.BTensor.from_parts(ctx, (0,), [[k], [3]], [[(0,)]] * 2, (0,), {(0, 0): v})
    out = qa.BTensor.from_parts(ctx, (0,), [[i], [j], [3]], [[(0,)]] * 3, (0,), {(0, 0, 0): np.zeros((i, j, 3))})
    a.tensordot_into(b, [1], [0], out)
    assert np.array_equal(from_dev(out).blocks[(0, 0, 0)], np.matmul(x.transpose(0, 2, 1), v))
