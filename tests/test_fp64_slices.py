"""FP64 slice contraction at the edges of its tasks.

Tasks longer than the records a workgroup holds in LDS (64) need an iteration with many slices
and a large task size; at the default size the same applies run in tasks of at most 64.  The
sums differ only in where a node's slices are cut into tasks, so the coefficients agree to
FP64 rounding: about 2000 terms per coefficient of at most the largest magnitude,
sqrt(2000) 1.1e-16 < 1e-14 of it typically, 1e-12 as for every other comparison of schedules.
The orders with one workgroup shape each (k = 3 to 7: rows split over 2, 3, 3, 4 and 4 waves;
k = 8 and 9: planes) run against the oracle with tasks of one, a few and many slices.
"""
import numpy as np
import pytest

from mrchem_amd import configs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    from mrchem_amd import mrcpp
    mrcpp.default_context()
    return mrcpp


@pytest.mark.parametrize("k,n_orb", [(7, 6), (9, 10)])
def test_tasks_longer_than_the_record_batch(G, k, n_orb):
    prec = 1e-6
    mra = G.mra_from(configs.BOX20, k)
    orbs, nuc, mus = configs.orbitals(7, n_orb=n_orb)
    trees = [G.project(prec, G.FunctionTree(mra), o) for o in orbs]
    ops = [G.HelmholtzOperator(mra, mu, prec) for mu in mus]
    saved = mra.ctx.get_tuning()
    try:
        res = []
        for chunk in (64, 4096):
            mra.ctx.set_tuning(chunk, saved[1])
            outs = [G.FunctionTree(mra) for _ in trees]
            G.apply_batch(prec, outs, ops, trees)
            res.append([o.export() for o in outs])
        for (d0, l0, c0), (d1, l1, c1) in zip(*res):
            assert np.array_equal(d0, d1) and np.array_equal(l0, l1)
            assert np.abs(c0 - c1).max() <= 1e-12 * np.abs(c0).max()
    finally:
        mra.ctx.set_tuning(*saved)


@pytest.mark.parametrize("basis", ["L", "I"])
@pytest.mark.parametrize("k", [3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("chunk", [1, 3, 64])
def test_every_order_against_the_oracle(G, k, basis, chunk):
    from oracle import mwref as M
    prec = 1e-3
    g, _ = configs.density3(4)
    mra = G.mra_from(configs.BOX16, k, basis)
    omra = M.MRA(**configs.BOX16, k=k, basis=basis, max_depth=16)
    of = M.Tree(omra).project_gauss(prec, g)
    f = G.FunctionTree(mra).load(*of.export())
    saved = mra.ctx.get_tuning()
    try:
        mra.ctx.set_tuning(chunk, saved[1])
        out = G.FunctionTree(mra)
        st = G.apply(prec, out, G.PoissonOperator(mra, prec), f)
    finally:
        mra.ctx.set_tuning(*saved)
    oout = M.Tree(omra)
    ost = M.apply(prec, oout, M.poisson(omra, prec), of)
    assert st["tuples"] == ost["tuples"] and st["nodes_out"] == ost["nodes_out"]
    c1, c2 = out.export()[2], oout.export()[2]
    assert np.abs(c1 - c2).max() <= 1e-12 * np.abs(c2).max()
