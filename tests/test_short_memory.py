"""Calls on a card whose memory is nearly used up.

A batch of products that fits at its own size runs, whatever ran on the context before it.  Most of
the card is held by an allocation that no kernel touches; the calls that run out of memory fail
on the host, in the allocator.
"""
import ctypes as C
import gc

import numpy as np
import pytest

from mrchem_amd import configs

pytestmark = pytest.mark.gpu

GIB = 1 << 30


class _Held:
    """All of the card's free memory but `left` bytes, through the HIP runtime that the library uses."""

    def __init__(self, ctx, left):
        from mrchem_amd import mrcpp
        gc.collect()
        for c in (ctx, mrcpp.default_context()):  # (the blocks that other tests left would be used first)
            c.trim()
        with open("/proc/self/maps") as f:
            paths = sorted({line.split()[-1] for line in f if "libamdhip64" in line})
        free, total, self.p = C.c_size_t(), C.c_size_t(), C.c_void_p()
        self.hip = next(h for h in map(C.CDLL, paths) if h.hipMemGetInfo(C.byref(free), C.byref(total)) == 0)
        assert self.hip.hipMalloc(C.byref(self.p), C.c_size_t(max(free.value - left, 1 << 20))) == 0

    def free(self):
        self.hip.hipFree(self.p)


def _products(G, mra, fine, n):
    outs = [G.FunctionTree(mra) for _ in range(n)]
    G.multiply_batch(0.5, outs, 1.0, [fine] * n, [fine] * n)
    return outs


def test_products_after_products_that_grew():
    from mrchem_amd import mrcpp as G
    ctx = G.Context(0)
    mra = G.mra_from(configs.BOX20, 9, ctx=ctx)
    orbs, _, _ = configs.orbitals(3, n_orb=2)
    coarse = G.project(0.3, G.FunctionTree(mra), orbs[0])
    fine = G.project(1e-8, G.FunctionTree(mra), orbs[0])
    one = _products(G, mra, fine, 1)[0]
    nodes = one.getNNodes()
    assert nodes == fine.getNNodes()  # (at this precision a product stays on the grid)
    n = int(2.4 * GIB / (nodes * 64000)) + 1
    grown = G.multiply(1e-6, G.FunctionTree(mra), 1.0, coarse, coarse)
    assert grown.getNNodes() > 2 * coarse.getNNodes()
    held = _Held(ctx, 4 * GIB)
    try:
        outs = _products(G, mra, fine, n)
        assert all(o.getNNodes() == nodes for o in outs)
        assert np.array_equal(outs[-1].export()[2], one.export()[2])
    finally:
        outs = None
        held.free()
        gc.collect()
        ctx.trim()


def test_outputs_of_a_call_that_runs_out_of_memory_are_empty():
    """(they would hold nodes without coefficients, which the next kernel reads)"""
    from mrchem_amd import mrcpp as G
    ctx = G.Context(0)
    mra = G.mra_from(configs.BOX20, 9, ctx=ctx)
    orbs, _, _ = configs.orbitals(3, n_orb=2)
    fine = G.project(1e-8, G.FunctionTree(mra), orbs[0])
    one = _products(G, mra, fine, 1)[0]
    n = int(2.4 * GIB / (one.getNNodes() * 64000)) + 1
    held = _Held(ctx, GIB)
    try:
        for call in (lambda o: G.multiply_batch(0.5, o, 1.0, [fine] * n, [fine] * n),
                     lambda o: G.add_batch(o, [[(1.0, fine)]] * n)):
            outs = [G.FunctionTree(mra) for _ in range(n)]
            with pytest.raises(G.MwgError, match="allocation"):
                call(outs)
            assert all(o.getNNodes() == 0 for o in outs)
            with pytest.raises(G.MwgError, match="empty"):
                G.add(G.FunctionTree(mra), 1.0, outs[0], 1.0, fine)
            outs = None
            gc.collect()
            ctx.trim()
    finally:
        held.free()
        gc.collect()
        ctx.trim()
    two = _products(G, mra, fine, 2)
    assert all(np.array_equal(t.export()[2], one.export()[2]) for t in two)
