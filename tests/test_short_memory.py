"""Products on a card whose memory is nearly used up.

A batch of products that fits at its own size runs, whatever ran on the context before it.  Most of
the card is held by an allocation that no kernel touches; the calls that run out of memory fail
on the host, in the allocator.
"""
import gc

import numpy as np
import pytest

from mrchem_amd import configs

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def _hold_all_but(ctx, left):
    import torch
    gc.collect()
    ctx.trim()
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    return torch.empty(max(free - left, 0), dtype=torch.uint8, device="cuda")


def _products(G, mra, fine, n):
    outs = [G.FunctionTree(mra) for _ in range(n)]
    G.multiply_batch(0.5, outs, 1.0, [fine] * n, [fine] * n)
    return outs


def test_products_after_products_that_grew():
    import torch
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
    held = _hold_all_but(ctx, 4 * GIB)
    try:
        outs = _products(G, mra, fine, n)
        assert all(o.getNNodes() == nodes for o in outs)
        assert np.array_equal(outs[-1].export()[2], one.export()[2])
    finally:
        outs = None
        del held
        torch.cuda.empty_cache()
        gc.collect()
        ctx.trim()
