"""Linear combinations whose records (output node, term) are many more than one launch takes.

The combinations of an orbital vector have a number of records that grows with its square; the
memory for them does not.  Sums of many terms over a few trees equal the sums with the terms'
coefficients added up first: n additions of at most sum |c| max |f| each, n 1.1e-16 of that.
"""
import threading
import time

import numpy as np
import pytest

from mrchem_amd import configs

pytestmark = pytest.mark.gpu


class _PeakMemory:
    """Growth of the process's resident memory while the block runs, in bytes."""

    def __enter__(self):
        self.base = self.peak = self._now()
        self.stop = threading.Event()
        self.t = threading.Thread(target=self._watch)
        self.t.start()
        return self

    @staticmethod
    def _now():
        with open("/proc/self/statm") as f:
            return 4096 * int(f.read().split()[1])

    def _watch(self):
        while not self.stop.is_set():
            self.peak = max(self.peak, self._now())
            time.sleep(0.0005)

    def __exit__(self, *a):
        self.stop.set()
        self.t.join()
        self.growth = self.peak - self.base


def _check(G, mra, f, sums, outs):
    for terms, o in zip(sums, outs):
        tot = [sum(c for c, t in terms if t is g) for g in f]
        ref = G.add_batch([G.FunctionTree(mra)], [list(zip(tot, f))])[0]
        (d0, l0, c0), (d1, l1, c1) = o.export(), ref.export()
        assert np.array_equal(d0, d1) and np.array_equal(l0, l1)
        scale = sum(abs(c) for c, _ in terms) * max(np.abs(t.export()[2]).max() for t in f)
        assert np.abs(c0 - c1).max() <= len(terms) * 1.2e-16 * scale
        assert abs(o.getSquareNorm() - ref.getSquareNorm()) <= 1e-12 * ref.getSquareNorm()


def test_memory_does_not_grow_with_the_number_of_records():
    from mrchem_amd import mrcpp as G
    mra = G.mra_from(configs.BOX20, 3)
    orbs, _, _ = configs.orbitals(4, n_orb=6)
    f = [G.project(p, G.FunctionTree(mra), o) for p, o in zip((1e-2, 3e-3, 1e-3, 1e-3, 1e-2, 1e-3), orbs)]
    nodes = max(t.getNNodes() for t in f)
    r = np.random.default_rng(1)

    def terms(m):
        return [(float(r.uniform(-1.0, 1.0)), f[i]) for i in list(range(len(f))) + list(r.integers(0, len(f), m - len(f)))]

    m = 256
    sums = [terms(m) for _ in range((10 << 20) // (nodes * m))]
    for n in (2, len(sums)):  # (the first call makes the buffers)
        outs = [G.FunctionTree(mra) for _ in range(n)]
        with _PeakMemory() as mem:
            G.add_batch(outs, sums[:n])
    _check(G, mra, f, sums[::7], outs[::7])
    # ten million records of 32 bytes on the host and 24 in the staging ring, or a million at a time
    assert mem.growth < 128 << 20
    # one combination beyond the bound, between small ones
    sums = [terms(7), terms((3 << 20) // nodes), terms(9)]
    outs = G.add_batch([G.FunctionTree(mra) for _ in sums], sums)
    _check(G, mra, f, sums, outs)
