"""The task sizes that are set are the ones that run, whatever ran on the context before.

Where a node's slices are cut into tasks shows in the last bits of its coefficients, and only
there: equal sizes give equal bits, other sizes other bits and values that agree to FP64
rounding (1e-12 of the largest coefficient, as for every comparison of schedules).
"""
import numpy as np
import pytest

from mrchem_amd import configs

pytestmark = pytest.mark.gpu


def _batch(k, prec, n_orb):
    """A context of its own and a function that applies the batch with the given task size."""
    from mrchem_amd import mrcpp as G
    ctx = G.Context(0)
    mra = G.mra_from(configs.BOX20, k, ctx=ctx)
    orbs, nuc, mus = configs.orbitals(7, n_orb=n_orb)
    trees = [G.project(prec, G.FunctionTree(mra), o) for o in orbs]
    ops = [G.HelmholtzOperator(mra, mu, prec) for mu in mus]

    def run(chunk, slice_chunk=0, flags=G.MWG_APPLY_FP64):
        ctx.set_tuning(chunk, slice_chunk)
        outs = [G.FunctionTree(mra) for _ in trees]
        st = G.apply_batch(prec, outs, ops, trees, flags=flags)
        return [o.export() for o in outs], all(s["device_loop"] == 1 for s in st)

    return run


def _same_bits(x, y):
    return all(np.array_equal(p, q) for a, b in zip(x, y) for p, q in zip(a, b))


def _close(x, y):
    for (d0, l0, c0), (d1, l1, c1) in zip(x, y):
        assert np.array_equal(d0, d1) and np.array_equal(l0, l1)
        assert np.abs(c0 - c1).max() <= 1e-12 * np.abs(c0).max()


@pytest.mark.parametrize("k,mixed", [(5, False), (9, False), (9, True)])
def test_a_smaller_size_is_used_after_a_larger_one(k, mixed):
    from mrchem_amd import mrcpp as G
    flags = G.MWG_APPLY_MIXED if mixed else G.MWG_APPLY_FP64
    sizes = (3, 5) if mixed else (3, 0)
    fresh, used = _batch(k, 1e-4, 2), _batch(k, 1e-4, 2)
    for _ in range(2):  # (the second on the device loop)
        want, dl = fresh(*sizes, flags)
    assert dl
    for _ in range(2):
        large, _ = used(4096, 4096 if mixed else 0, flags)
    for _ in range(2):
        got, dl = used(*sizes, flags)
    assert dl
    assert not _same_bits(want, large)
    assert _same_bits(want, got)
    _close(large, got)


@pytest.mark.parametrize("k", [4, 6, 7, 8, 9])
def test_tasks_of_more_than_two_record_batches(k):
    """A workgroup holds 64 records at a time.  The largest size differs from 128 in its bits, so
    some task has more than 128 records."""
    run = _batch(k, 10.0 ** -min(k - 1, 6), 12 if k >= 6 else 24)
    for _ in range(2):
        a, _ = run(128)
    for _ in range(2):
        b, _ = run(4096)
    assert not _same_bits(a, b)
    _close(a, b)
