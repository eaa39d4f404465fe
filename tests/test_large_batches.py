"""Batches beyond the sizes at which the host's bookkeeping and the operator build change.

Trees of more than 65536 nodes in a batch are handled on host threads (union grids, item lists, node
tables, input scans); operator levels whose child-scale rows exceed 256 MiB are built in several
chunks (at k = 9 about 170 operators of precision 1e-6).  The results are those of single calls.
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


def _same_bits(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a.export(), b.export()))


def _close(a, b):
    (d0, l0, c0), (d1, l1, c1) = a.export(), b.export()
    assert np.array_equal(d0, d1) and np.array_equal(l0, l1)
    assert np.abs(c0 - c1).max() <= 1e-12 * np.abs(c0).max()


def test_bookkeeping_on_threads(G):
    """Products and sums of a batch equal single calls to the bit; applies to FP64 rounding (their
    tasks are cut by the batch's slices)."""
    prec = 1e-3
    mra = G.mra_from(configs.BOX20, 3)
    orbs, _, _ = configs.orbitals(4, n_orb=6)
    f = [G.project(prec, G.FunctionTree(mra), o) for o in orbs]
    reps = 70000 // sum(t.getNNodes() for t in f) + 1
    a, b = f * reps, (f[1:] + f[:1]) * reps
    prods = G.multiply_batch(prec, [G.FunctionTree(mra) for _ in a], 1.0, a, b)
    sums = G.add_batch([G.FunctionTree(mra) for _ in a], [[(0.5, x), (-2.0, y)] for x, y in zip(a, b)])
    assert sum(t.getNNodes() for t in prods) > 65536
    P = G.PoissonOperator(mra, prec)
    for _ in range(2):  # (the second on the device loop)
        pots = [G.FunctionTree(mra) for _ in prods]
        G.apply_batch(prec, pots, [P] * len(prods), prods)
    for i in range(6):
        p = G.multiply(prec, G.FunctionTree(mra), 1.0, a[i], b[i])
        s = G.add(G.FunctionTree(mra), 0.5, a[i], -2.0, b[i])
        v = G.FunctionTree(mra)
        G.apply(prec, v, P, p)
        for j in range(i, len(prods), 6):
            assert _same_bits(prods[j], p) and _same_bits(sums[j], s)
            _close(pots[j], v)


def test_operator_levels_in_several_chunks(G):
    """The levels of 220 new operators, built for one batch, against one operator at a time."""
    prec = 1e-3
    mra = G.mra_from(configs.BOX20, 9)
    t = G.project(prec, G.FunctionTree(mra), configs.orbitals(1, n_orb=1)[0][0])
    mus = [0.3 + 0.01 * i for i in range(220)]
    outs = [G.FunctionTree(mra) for _ in mus]
    G.apply_batch(prec, outs, [G.HelmholtzOperator(mra, mu, 1e-6) for mu in mus], [t] * len(mus))
    for i in range(0, len(mus), 9):
        o = G.FunctionTree(mra)
        G.apply(prec, o, G.HelmholtzOperator(mra, mus[i], 1e-6), t)
        _close(outs[i], o)
